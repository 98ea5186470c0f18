// qb_rayref.hip -- gfx950 kernels of the reference's own float trajectory (anneal_branch,
// src/ising_recon.hpp:119-143): ray_ref_kernel, and ray_ref_lane_kernel for many branches of short
// columns.
//
// Branch b anneals from x = 0, r = -d with seed b + 1 + seed_offset: bits in index order,
// dE = local_field_dE (lin delta, then w (r a + a^2 / 2) per entry with a = a_k delta in CSR
// order, then lambda (+-1) per neighbour in CSR order), one splitmix64 stream drawn only
// for uphill proposals, a flip iff dE <= 0 or u < exp(-dE / T), and on a flip r += a_k delta
// per entry. Draw keys and counters of unions (draw_bit, draw_key) do not apply here.
#include <algorithm>

#include "qb_internal.h"
#include "qb_rng.h"

namespace qb {

namespace {

using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
using i32x4 = int32_t __attribute__((ext_vector_type(4)));
using f32x4 = float __attribute__((ext_vector_type(4)));
using f64x2 = double __attribute__((ext_vector_type(2)));

constexpr int kQuads = 3;               // four entries of a lane each, in flight
constexpr int kBatch = 256 * kQuads;    // entries of a batch
constexpr int kPassBatches = 5;         // batches of one pass at most, its terms in LDS
constexpr int kTail = 16;               // terms a lane reads ahead of its sum
constexpr int kNb = kRefNb;             // neighbours of a bit held in registers; more are read in turn
static_assert(2 * kBatch <= kRefPad && kNb == 8);

__device__ __forceinline__ double flip_sign(double v, uint32_t bit) {
    return __hiloint2double(__double2hiint(v) ^ int(bit << 31), __double2loint(v));
}

// A wave anneals one branch; its spins are a bit mask in LDS (LDS_X), or bytes in global
// memory where the mask does not fit beside the terms, its residuals FP64 in global memory.
// The wave takes the bits 64 at a time, a lane each.
//
// The window's columns lie one after the other (RefLayout). The wave computes their terms
// entry by entry, 64 at a time whatever the columns' lengths, into LDS, and each lane then adds
// its own column's terms, in order. Then the window's decisions are found by iteration: with a
// guess of the window's flips, every lane sums its neighbour terms on the spins that the guess
// leaves before it, is downhill or uphill, takes the draw that the uphill lanes before it leave
// it, and decides. Decisions depend on earlier lanes only, so those up to the first lane where
// the outcome differs from the guess are the loop's own; the outcome is the next guess. Where
// a bit with rays flips, the lanes up to it stand, the residuals are updated and the later
// lanes' columns are summed again.
//
// 1,024 branches of the muon QUBO on a 32^3 grid (5,028 bits, 75,938 entries, 6,000 rays), 50
// sweeps from T = 50 to 1: 22 ms, where a lane that walks its own column and ends the window
// at every flip takes 215 (a round trip to memory per flip and per eight entries). A sweep is
// bound by one wave's instructions, a branch having a SIMD to itself: at T = 1, 565 thousand
// cycles, 240 for the terms (116 batches, 250 instructions and the L1's 20 KB each), 112 for the
// ordered sums (5,200 dependent additions), 140 for the windows' neighbours and draws and 70
// for the decisions; at T = 50, where 200 bits with rays flip, 2 million. A batch whose
// loads are waited for where they are issued costs 1.3 times as much, three separate loads an
// entry 1.1 times.
//
// A launch runs sweeps [sweep_begin, sweep_end); the first one starts every branch from
// x = 0, r = -d and its seed's splitmix64 state, a later one continues from the x, r and
// state (sm[b]) the previous launch left, so the split never changes the trajectory.
template <bool LDS_X>
__global__ void __launch_bounds__(64) ray_ref_kernel(DevProblem p, uint64_t seed_offset, const double* temp,
                                                      int sweep_begin, int sweep_end, uint8_t* xs, double* rs,
                                                      uint64_t* sm, int pass) {
    extern __shared__ __align__(16) double terms[];   // pass terms, and what a lane reads past them
    // LDS_X: bit i of the branch is bit i % 64 of word i / 64
    uint64_t* xw = reinterpret_cast<uint64_t*>(terms + pass + 2 * kTail);
    const int lane = int(threadIdx.x), b = int(blockIdx.x);
    const int n = p.n, n_win = (n + 63) / 64;
    uint8_t* x = xs + size_t(b) * size_t(n);
    double* r = rs + size_t(b) * size_t(p.n_rays);
    uint64_t st;
    if (sweep_begin == 0) {
        if constexpr (LDS_X) {
            for (int w = lane; w < n_win; w += 64) xw[w] = 0;
        } else {
            for (int i = lane; i < n; i += 64) x[i] = 0;
        }
        for (int k = lane; k < p.n_rays; k += 64) r[k] = -p.d[k];
        st = (uint64_t(b) + 1u + seed_offset) * 0x2545F4914F6CDD1Dull + 1;
    } else {
        st = sm[b];
        if constexpr (LDS_X)
            for (int w = 0; w < n_win; ++w) {
                const int i = w * 64 + lane;
                const uint64_t word = __ballot(i < n && x[i < n ? i : 0] != 0);
                if (lane == 0) xw[w] = word;
            }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
    auto spin = [&](int i) -> uint32_t {
        if constexpr (LDS_X) return (reinterpret_cast<const uint32_t*>(xw)[i >> 5] >> (i & 31)) & 1u;
        else return x[i];
    };
    const uint64_t below = (uint64_t(1) << lane) - 1u;
    // what a window needs of its lanes' bits, read one window ahead
    struct Bit {
        u32x4 at;     // RefBit
        u32x4 base;   // RefBase
        i32x4 nb[kNb / 4];
    };
    auto load_bit = [&](int win) {
        const int i = min(win * 64 + lane, n - 1);
        Bit v;
        v.at = *reinterpret_cast<const u32x4*>(p.ref.bit + i);
        v.base = *reinterpret_cast<const u32x4*>(p.ref.base + i);
#pragma unroll
        for (int k = 0; k < kNb / 4; ++k) v.nb[k] = reinterpret_cast<const i32x4*>(p.ref.nb + size_t(i) * kNb)[k];
        return v;
    };
    Bit cur{};
    if (n_win > 0 && sweep_begin < sweep_end) cur = load_bit(0);
    // a batch of kBatch entries, read before it is asked for: its fields and residuals from
    // entry held, the rays of the batch after it from entry held_rays. In a block of 256 entries a
    // lane has entries lane, lane + 64, lane + 128 and lane + 192.
    u32x4 ray[kQuads];
    uint32_t own[kQuads];
    f32x4 a[kQuads];
    f64x2 w[kQuads][2];
    double rv[kQuads][4];
    uint64_t held = ~uint64_t(0), held_rays = ~uint64_t(0);   // multiples of 256 where they stand for a batch
    const unsigned quad = unsigned(lane) * 4u;
    auto load_rays = [&](int v, uint64_t at) {
        ray[v] = *reinterpret_cast<const u32x4*>(p.ref.ray + (at + 256u * v) + quad);
    };
    auto load_fields = [&](int v, uint64_t at) {
        own[v] = *reinterpret_cast<const uint32_t*>(p.ref.own + (at + 256u * v) + quad);
        a[v] = *reinterpret_cast<const f32x4*>(p.ref.a + (at + 256u * v) + quad);
        const double* q = p.ref.w + (at + 256u * v) + quad;
        w[v][0] = *reinterpret_cast<const f64x2*>(q);
        w[v][1] = *reinterpret_cast<const f64x2*>(q + 2);
    };
    auto load_residuals = [&](int v) {
#pragma unroll
        for (int u = 0; u < 4; ++u) rv[v][u] = r[ray[v][u]];
    };
    for (int sweep = sweep_begin; sweep < sweep_end; ++sweep) {
        const double T = temp[sweep];
        const double nrT = T < 1e300 ? -1.0 / T : __builtin_nan("");   // NaN: every exponential exact
        for (int win = 0; win < n_win; ++win) {
            Bit next = load_bit(win + 1 < n_win ? win + 1 : 0);
            const int i0 = win * 64, i = i0 + lane;
            const bool valid = i < n;
            const uint64_t vmask = __ballot(valid);
            const unsigned c0 = cur.at.x, c1 = cur.at.y, nnb = valid ? cur.at.z & 0x7FFFFFFFu : 0u;
            const bool heavy = valid && c1 > c0;
            const uint64_t hmask = __ballot(heavy);
            const uint32_t xi = valid ? spin(i) : 0u;
            const int n_terms = __ballot(nnb > 6u) ? 8 : __ballot(nnb > 4u) ? 6 : 4;
            // a neighbour's term on the spins before the window, and the shift that brings its
            // flip to bit 0 if it comes earlier in the window (the lane's own bit, masked out
            // below, if not)
            uint32_t xn[kNb];
            double term[kNb];
            int shift[kNb];
#pragma unroll
            for (int k = 0; k < kNb; ++k) xn[k] = spin(cur.nb[k / 4][k % 4]);
#pragma unroll
            for (int k = 0; k < kNb; ++k) {
                if (k >= n_terms) break;
                const double t = flip_sign(p.lambda, xn[k] ^ xi);
                term[k] = unsigned(k) < nnb ? t : -0.0;
                const int d = cur.nb[k / 4][k % 4] - i0;
                shift[k] = unsigned(d) < 64u ? d : lane;
            }
            const bool longer = __ballot(nnb > unsigned(kNb)) != 0;
            const double u_mine = double(mix64(st + uint64_t(lane + 1) * kGamma) >> 11) * 0x1.0p-53;

            uint64_t flips = 0, todo = vmask;
            int drawn = 0;
            const double lin = __hiloint2double(int(cur.base.y), int(cur.base.x));
            const double plain = xi ? -lin : lin;   // the sum up to the column
            const uint64_t xmask = __ballot(xi != 0);
            double col = plain;
            const uint64_t base = uint64_t(unsigned(__builtin_amdgcn_readlane(int(cur.base.z), 0))) |
                                  uint64_t(unsigned(__builtin_amdgcn_readlane(int(cur.base.w), 0))) << 32;
            const unsigned len = unsigned(__builtin_amdgcn_readlane(int(c1), 63 - __builtin_clzll(vmask)));
            const uint64_t end = base + ((len + 255u) & ~255u);
            uint64_t from = base;
            for (;;) {
                for (uint64_t p0 = from, p1; p0 < end; p0 = p1) {
                    p1 = end - p0 > uint64_t(pass) ? p0 + uint64_t(pass) : end;
                    if (held != p0) {   // in the loop's order, so that its waits fit both
#pragma unroll
                        for (int v = 0; v < kQuads; ++v) load_rays(v, p0);
                        held_rays = p0 + kBatch;
#pragma unroll
                        for (int v = 0; v < kQuads; ++v) {
                            __builtin_amdgcn_sched_barrier(0);
                            load_residuals(v);
                            load_rays(v, held_rays);
                            load_fields(v, p0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    for (uint64_t g = p0, then; g < p1; g = then) {
                        then = p1 - g > kBatch ? g + kBatch : p1;
                        if (held_rays != then) {
#pragma unroll
                            for (int v = 0; v < kQuads; ++v) load_rays(v, then);
#pragma unroll
                            for (int v = 0; v < kQuads; ++v) asm volatile("" : "+v"(ray[v]));   // waits here
                        }
#pragma unroll
                        for (int v = 0; v < kQuads; ++v) {
                            __builtin_amdgcn_sched_barrier(0);
                            if (int(p1 - g) > 256 * v) {   // the batch's last blocks may be empty
                                // a is a float's value, so 0.5 a a is exact and the fused add rounds
                                // as the separate one does; four entries side by side, as the wave
                                // has its SIMD to itself and each step's result takes a while
                                double ad[4], t[4];
#pragma unroll
                                for (int u = 0; u < 4; ++u) ad[u] = double(a[v][u]);
                                uint32_t neg[4];
#pragma unroll
                                for (int u = 0; u < 4; ++u) neg[u] = uint32_t(xmask >> ((own[v] >> (8 * u)) & 63u)) << 31;
                                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                                for (int u = 0; u < 4; ++u)
                                    ad[u] = __hiloint2double(__double2hiint(ad[u]) ^ int(neg[u]), __double2loint(ad[u]));
                                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                                for (int u = 0; u < 4; ++u) t[u] = rv[v][u] * ad[u];
                                double half[4];
#pragma unroll
                                for (int u = 0; u < 4; ++u) half[u] = 0.5 * ad[u];
                                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                                for (int u = 0; u < 4; ++u) t[u] = __builtin_fma(half[u], ad[u], t[u]);
                                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                                for (int u = 0; u < 4; ++u) t[u] *= w[v][u / 2][u % 2];
                                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                                for (int u = 0; u < 4; ++u) terms[int(g - p0) + 256 * v + 64 * u + lane] = t[u];
                            }
                            __builtin_amdgcn_sched_barrier(0);
                            load_residuals(v);
                            load_rays(v, then + kBatch);
                            load_fields(v, then);
                        }
                        held = then;
                        held_rays = then + kBatch;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    const unsigned r0 = unsigned(p0 - base), r1 = unsigned(p1 - base);
                    const unsigned k0 = max(c0, r0) - r0;
                    int left = int(min(c1, r1) - r0) - int(k0);
                    if (heavy && ((todo >> lane) & 1u) && left > 0) {
                        const double* t = terms + k0;
                        double v[kTail];
#pragma unroll
                        for (int u = 0; u < kTail; ++u) v[u] = t[u];
                        for (; left >= kTail; left -= kTail) {
                            t += kTail;
#pragma unroll
                            for (int u = 0; u < kTail; ++u) {
                                col += v[u];
                                v[u] = t[u];
                            }
                        }
#pragma unroll
                        for (int u = 0; u < kTail; ++u) {
                            if (u % 4 == 0 && __ballot(u < left) == 0) break;
                            col += u < left ? v[u] : -0.0;
                        }
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                }
                uint64_t guess = flips, up_mask, taken, h;
                for (;;) {
                    const uint64_t before = guess & below;
                    double dE = col;
#pragma unroll
                    for (int k = 0; k < kNb; ++k) {
                        if (k >= n_terms) break;
                        dE += flip_sign(term[k], uint32_t(before >> shift[k]));
                    }
                    if (longer)
                        for (unsigned q = cur.at.w + kNb; q < cur.at.w + nnb; ++q) {
                            const int nb = p.nb_bit[q];
                            const int s = unsigned(nb - i0) < 64u ? nb - i0 : lane;
                            dE += flip_sign(p.lambda, spin(nb) ^ xi ^ uint32_t(before >> s));
                        }
                    const bool up = dE > 0.0;
                    up_mask = __ballot(up) & todo;
                    const double u = __shfl(u_mine, drawn + __popcll(up_mask & below));
                    bool take = dE <= 0.0;
                    if (up) take = ref_accept_u(u, dE, T, nrT);
                    taken = __ballot(take) & todo;
                    const uint64_t outcome = flips | taken, wrong = outcome ^ guess;
                    h = taken & hmask;
                    if (wrong == 0 || (h != 0 && __builtin_ctzll(h) <= __builtin_ctzll(wrong))) break;
                    guess = outcome;
                }
                if (h == 0) {
                    flips |= taken;
                    drawn += __popcll(up_mask);
                    break;
                }
                const int js = __builtin_ctzll(h);
                const uint64_t upto = js == 63 ? ~uint64_t(0) : (uint64_t(2) << js) - 1u;
                flips |= taken & upto;
                drawn += __popcll(up_mask & upto);
                todo = vmask & ~upto;
                const unsigned k0 = unsigned(__builtin_amdgcn_readlane(int(c0), js));
                const unsigned k1 = unsigned(__builtin_amdgcn_readlane(int(c1), js));
                const uint32_t neg = uint32_t(__builtin_amdgcn_readlane(int(xi), js));
                if (!(__builtin_amdgcn_readlane(int(cur.at.z), js) < 0)) {
                    for (unsigned k = k0 + unsigned(lane); k < k1; k += 64) {
                        const uint64_t at = ref_slot(base + k);
                        r[p.ref.ray[at]] += flip_sign(double(p.ref.a[at]), neg);
                    }
                } else if (lane == 0) {   // a ray repeats in the column: its additions in CSR order
                    for (unsigned k = k0; k < k1; ++k) {
                        const uint64_t at = ref_slot(base + k);
                        r[p.ref.ray[at]] += flip_sign(double(p.ref.a[at]), neg);
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
                __builtin_amdgcn_wave_barrier();
                held = ~uint64_t(0);   // its residuals may have changed
                if (todo == 0) break;
                from = base + (k1 & ~255u);
                col = heavy ? plain : col;
            }
            st += uint64_t(drawn) * kGamma;
            if (flips != 0) {
                if constexpr (LDS_X) {
                    if (lane == 0) xw[win] ^= flips;
                } else {
                    if ((flips >> lane) & 1u) x[i] = uint8_t(xi ^ 1u);
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
                __builtin_amdgcn_wave_barrier();
            }
            cur = next;
        }
    }
    if constexpr (LDS_X)
        for (int i = lane; i < n; i += 64) x[i] = uint8_t((xw[i >> 6] >> (i & 63)) & 1u);
    if (lane == 0) sm[b] = st;
}

// Many branches of short columns: a lane walks its own bit's column, eight entries' loads in flight,
// and the first accepted bit of a window is the loop's next flip. A flip of a bit with rays ends
// the window; after a ray-free bit's flip the later lanes only sum their neighbour terms again
// and decide anew. Spins are bytes in global memory. ray_ref_kernel's registers hold a CU to eight of
// its waves; this one's leave room for 28, whose round trips to memory overlap, and a column of a few
// entries is one such trip: 4,096 branches of 200 bits with three entries each, 20 sweeps at T = 20, take
// 24.4 ms here and 32.3 there (16 branches 10.7 and 6.4). Where the line lies: ref_lane_from.
__global__ void __launch_bounds__(256) ray_ref_lane_kernel(DevProblem p, int R, uint64_t seed_offset, const double* temp,
                                                           int sweep_begin, int sweep_end, uint8_t* xs, double* rs,
                                                           uint64_t* sm) {
    const int w = int(threadIdx.x) / 64, lane = int(threadIdx.x) % 64;
    const int b = int(blockIdx.x) * 4 + w;
    if (b >= R) return;   // the whole wave leaves; waves never sync with each other
    const int n = p.n;
    uint8_t* x = xs + size_t(b) * size_t(n);
    double* r = rs + size_t(b) * size_t(p.n_rays);
    uint64_t st;
    if (sweep_begin == 0) {
        for (int i = lane; i < n; i += 64) x[i] = 0;
        for (int k = lane; k < p.n_rays; k += 64) r[k] = -p.d[k];
        st = (uint64_t(b) + 1u + seed_offset) * 0x2545F4914F6CDD1Dull + 1;
    } else {
        st = sm[b];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
    const uint64_t below = (uint64_t(1) << lane) - 1u;
    for (int sweep = sweep_begin; sweep < sweep_end; ++sweep) {
        const double T = temp[sweep];
        const double nrT = T < 1e300 ? -1.0 / T : __builtin_nan("");   // NaN: every exponential exact
        int i0 = 0;
        while (i0 < n) {
            const int i = i0 + lane;
            const bool valid = i < n;
            const int pos = valid ? p.bit_pos[i] : 0;
            double dE = 0.0, base = 0.0;   // base: the sum up to the neighbour terms
            const int xi = valid ? int(x[i]) : 0;
            // each lane's column bounds and update order, kept for the flip
            const int c0 = valid ? p.col_ptr[pos] : 0, c1 = valid ? p.col_ptr[pos + 1] : 0;
            const int seq = valid ? int(p.seq_update[pos]) : 0;
            constexpr int kChunk = 8;
            if (valid) {
                // eight entries' loads, then their residuals, in flight together; the sum
                // itself stays in CSR order
                const double delta = xi ? -1.0 : 1.0;
                dE = p.lin[pos] * delta;
                const int k1 = c1;
                for (int kb = c0; kb < k1; kb += kChunk) {
                    RayEnt e[kChunk];
                    double rv[kChunk];
#pragma unroll
                    for (int u = 0; u < kChunk; ++u) e[u] = p.ent[min(kb + u, k1 - 1)];
#pragma unroll
                    for (int u = 0; u < kChunk; ++u) rv[u] = r[e[u].ray];
#pragma unroll
                    for (int u = 0; u < kChunk; ++u) {
                        if (kb + u >= k1) break;
                        const double a = double(e[u].a) * delta;
                        dE += e[u].w * (rv[u] * a + 0.5 * a * a);
                    }
                }
                base = dE;
                const int q1 = p.nb_ptr[pos + 1];
                for (int qb = p.nb_ptr[pos]; qb < q1; qb += kChunk) {
                    int xv[kChunk];
#pragma unroll
                    for (int u = 0; u < kChunk; ++u) xv[u] = x[p.nb_bit[min(qb + u, q1 - 1)]];
#pragma unroll
                    for (int u = 0; u < kChunk; ++u) {
                        if (qb + u >= q1) break;
                        dE += p.lambda * (xv[u] != xi ? -1.0 : 1.0);
                    }
                }
            }
            // decisions of the lanes in todo (lanes >= lo) on the current state, the k-th
            // uphill one drawing st + k gamma
            uint64_t todo = ~uint64_t(0), m_up = 0, m_acc = 0;
            auto decide = [&]() {
                const bool mine = valid && ((todo >> lane) & 1u);
                const bool up = mine && dE > 0.0;
                m_up = __ballot(up) & todo;
                bool acc = mine && dE <= 0.0;
                if (up) acc = ref_accept(mix64(st + uint64_t(__popcll(m_up & below) + 1) * kGamma) >> 11, dE, T, nrT);
                m_acc = __ballot(acc) & todo;
            };
            decide();
            for (;;) {
                if (m_acc == 0) {
                    st += uint64_t(__popcll(m_up)) * kGamma;
                    i0 += 64;
                    break;
                }
                const int js = __builtin_ctzll(m_acc);
                const uint64_t upto = js == 63 ? ~uint64_t(0) : (uint64_t(2) << js) - 1u;
                st += uint64_t(__popcll(m_up & upto)) * kGamma;
                const int fi = i0 + js;
                const int k0 = __shfl(c0, js), k1 = __shfl(c1, js), seq_f = __shfl(seq, js);
                const int xf = __shfl(xi, js);
                const double delta = xf ? -1.0 : 1.0;
                if (!seq_f) {
                    for (int k = k0 + lane; k < k1; k += 64) r[p.ent[k].ray] += double(p.ent[k].a) * delta;
                } else if (lane == 0) {   // a ray repeats in the column: its additions in CSR order
                    for (int k = k0; k < k1; ++k) r[p.ent[k].ray] += double(p.ent[k].a) * delta;
                }
                if (lane == 0) x[fi] = uint8_t(xf ^ 1);
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
                __builtin_amdgcn_wave_barrier();
                todo = ~upto;
                if (k1 > k0 || todo == 0) {   // residuals changed (or the window is done)
                    i0 = fi + 1;
                    break;
                }
                // A ray-free bit flipped: no residual changed, so a later lane's sum up to its
                // neighbour terms stands; only those terms are summed again, in order.
                if (valid && ((todo >> lane) & 1u)) {
                    dE = base;
                    const int q1 = p.nb_ptr[pos + 1];
                    for (int qb = p.nb_ptr[pos]; qb < q1; qb += kChunk) {
                        int xv[kChunk];
#pragma unroll
                        for (int u = 0; u < kChunk; ++u) xv[u] = x[p.nb_bit[min(qb + u, q1 - 1)]];
#pragma unroll
                        for (int u = 0; u < kChunk; ++u) {
                            if (qb + u >= q1) break;
                            dE += p.lambda * (xv[u] != xi ? -1.0 : 1.0);
                        }
                    }
                }
                decide();
            }
        }
    }
    if (lane == 0) sm[b] = st;
}

// Zero entries: the layout's gaps and padding.
__global__ void __launch_bounds__(256) ref_zero_kernel(RefLayout to, size_t entries) {
    for (size_t k = size_t(blockIdx.x) * 256 + threadIdx.x; k < entries; k += size_t(gridDim.x) * 256) {
        to.ray[k] = 0;
        to.a[k] = 0.0f;
        to.w[k] = 0.0;
        to.own[k] = 0;
    }
}

// The bits and their columns in bit order, one wave a bit.
__global__ void __launch_bounds__(256) ref_layout_kernel(DevProblem p, RefLayout to) {
    const int i = int(blockIdx.x) * 4 + int(threadIdx.x) / 64, lane = int(threadIdx.x) % 64;
    if (i >= p.n) return;
    const int pos = p.bit_pos[i], k0 = p.col_ptr[pos], len = p.col_ptr[pos + 1] - k0;
    const int q0 = p.nb_ptr[pos], nnb = p.nb_ptr[pos + 1] - q0;
    const uint64_t at = p.ref_start[i], base = p.ref_start[i & ~63];
    for (int k = lane; k < len; k += 64) {
        const RayEnt e = p.ent[k0 + k];
        const uint64_t slot = ref_slot(at + unsigned(k));
        to.ray[slot] = uint32_t(e.ray);
        to.a[slot] = e.a;
        to.w[slot] = e.w;
        to.own[slot] = uint8_t(i & 63);
    }
    if (lane < kNb) to.nb[size_t(i) * kNb + size_t(lane)] = lane < nnb ? p.nb_bit[q0 + lane] : i;
    if (lane == 0) {
        to.bit[i] = RefBit{unsigned(at - base), unsigned(at - base) + unsigned(len),
                           unsigned(nnb) | (p.seq_update[pos] ? 0x80000000u : 0u), unsigned(q0)};
        to.base[i] = RefBase{p.lin[pos], base};
    }
}

}  // namespace

hipError_t launch_ref_layout(const DevProblem& p, const RefLayout& to, size_t entries, hipStream_t st) {
    ref_zero_kernel<<<unsigned(std::min<size_t>((entries + 255) / 256, 2048)), 256, 0, st>>>(to, entries);
    if (p.n > 0) ref_layout_kernel<<<unsigned((p.n + 3) / 4), 256, 0, st>>>(p, to);
    return hipGetLastError();
}

hipError_t launch_ray_ref_lane(const DevProblem& p, int R, uint64_t seed_offset, const double* temp, int sweep_begin,
                               int sweep_end, uint8_t* xs, double* rs, uint64_t* sm, hipStream_t st) {
    ray_ref_lane_kernel<<<unsigned((R + 3) / 4), 256, 0, st>>>(p, R, seed_offset, temp, sweep_begin, sweep_end, xs, rs,
                                                               sm);
    return hipGetLastError();
}

hipError_t launch_ray_ref(const DevProblem& p, int64_t widest, int R, uint64_t seed_offset, const double* temp, int sweep_begin,
                          int sweep_end, uint8_t* xs, double* rs, uint64_t* sm, hipStream_t st) {
    // a pass holds the widest window where it can: with fewer terms in LDS more branches share a
    // CU (4,096 branches of 100 bits and 500 entries, 20 sweeps at T = 20: 22.6 ms with five batches, 22.1
    // with one)
    const int pass = kBatch * int(std::clamp<int64_t>((widest + kBatch - 1) / kBatch, 1, kPassBatches));
    const size_t terms = sizeof(double) * size_t(pass + 2 * kTail);
    const size_t mask = sizeof(uint64_t) * ((size_t(p.n) + 63) / 64);
    if (mask <= 32768 - sizeof(double) * 2 * kTail)   // 260,096 bits; within 64 KiB with the terms
        ray_ref_kernel<true>
            <<<unsigned(R), 64, terms + mask, st>>>(p, seed_offset, temp, sweep_begin, sweep_end, xs, rs, sm, pass);
    else
        ray_ref_kernel<false>
            <<<unsigned(R), 64, terms, st>>>(p, seed_offset, temp, sweep_begin, sweep_end, xs, rs, sm, pass);
    return hipGetLastError();
}

}  // namespace qb
