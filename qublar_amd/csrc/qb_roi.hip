// qb_roi.hip -- gfx950 kernels of the exact region-of-interest posterior.
//
// A small QUBO E(x) = sum_i h_i x_i + sum_{i<j} J_ij x_i x_j over n <= 36 bits (the
// conditional QUBO of roi_qubo, src/ising_recon.hpp:245-300) is enumerated over all 2^n
// states, as tools/branches_blaze.py:45-53 does on the host: the minimum energy and its
// state, then Z = sum exp(-beta (E - E_min)) and every bit's weight sum_x w(x) x_i.
//
// The state index splits into low bits, kRoiThreadBits thread bits and block bits. The low
// bits are kRoiGroupBits group bits and B walked bits. A thread starts from the energy and
// the low bits' fields with its high bits set, walks the B bits in Gray order (one field
// update per step, of the low bits only; the flipped bit is the same in every lane, so its
// couplings are uniform), and at each step takes all 32 states of the group bits at once:
//   - their energies by doubling, E[2^a + s] = E[s] + (f_a + the couplings of a inside s), 57
//     additions;
//   - or their weights, W[2^a + s] = W[s] T_a[s] with T_a[0] = exp(-beta f_a) and a constant
//     factor exp(-beta J) per coupling inside the group: 6 exponentials for 32 states.
// The high bits' weights come from the sums of threads and blocks, once each.
//
// A carried field or energy has taken at most 2^B <= 128 steps, where walking every low bit
// in Gray order took 4,096, so energies are nearer a scratch sum. The walk that updated all
// n fields at every state and took an exponential for each state needed about 70 and 100
// vector instructions per state in the two passes; this needs about 4 and 10. A call with
// n = 26 takes 0.13 ms (2.07 before), with n = 32 2.1 ms (33.6 before: 2.0e12 states/s), with
// n = 36 26 ms.
//
// The bound is vector issue. Results depend on n and the inputs alone.
#include "qb_internal.h"

namespace qb {

constexpr int kRoiBlock = 1 << kRoiThreadBits;
constexpr int kRoiStates = 1 << kRoiGroupBits;

namespace {

// What a block shares: the fields of the low and thread bits with the block bits set.
template <int L>
struct RoiShared {
    double J[L][L];                     // among the low bits
    double JT[kRoiThreadBits][L];       // thread bit x low bit
    double JTT[kRoiThreadBits][kRoiThreadBits];
    double F[L], FT[kRoiThreadBits];
    double e;                           // the block bits' own energy
};

template <int L>
__device__ __forceinline__ void roi_stage(int n, const double* h, const double* Js, uint64_t block, RoiShared<L>& s) {
    constexpr int kHigh = L + kRoiThreadBits;   // first block bit
    const int t = int(threadIdx.x);
    for (int i = t; i < kHigh * kHigh; i += kRoiBlock) {
        const int r = i / kHigh, c = i % kHigh;
        const double v = Js[size_t(r) * size_t(n) + size_t(c)];
        if (r < L && c < L) s.J[r][c] = v;
        else if (r >= L && c < L) s.JT[r - L][c] = v;
        else if (r >= L) s.JTT[r - L][c - L] = v;
    }
    if (t < kHigh) {
        double f = h[t];
        for (int i = kHigh; i < n; ++i)
            if ((block >> (i - kHigh)) & 1u) f += Js[size_t(t) * size_t(n) + size_t(i)];
        if (t < L) s.F[t] = f;
        else s.FT[t - L] = f;
    } else if (t == 64) {
        double e = 0.0;
        for (int i = kHigh; i < n; ++i) {
            if (!((block >> (i - kHigh)) & 1u)) continue;
            double f = h[i];
            for (int j = kHigh; j < i; ++j)
                if ((block >> (j - kHigh)) & 1u) f += Js[size_t(i) * size_t(n) + size_t(j)];
            e += f;
        }
        s.e = e;
    }
    __syncthreads();
}

// A thread's walk: energy e and fields f of the low bits at the current Gray step.
template <int B>
struct RoiWalk {
    static constexpr int L = kRoiGroupBits + B;
    double e, f[L];

    __device__ __forceinline__ void start(const RoiShared<L>& s) {
        e = s.e;
#pragma unroll
        for (int j = 0; j < L; ++j) f[j] = s.F[j];
#pragma unroll
        for (int t = 0; t < kRoiThreadBits; ++t) {
            if (!((threadIdx.x >> t) & 1u)) continue;
            double ft = s.FT[t];
#pragma unroll
            for (int q = 0; q < t; ++q) ft += ((threadIdx.x >> q) & 1u) ? s.JTT[t][q] : 0.0;
            e += ft;
#pragma unroll
            for (int j = 0; j < L; ++j) f[j] += s.JT[t][j];
        }
    }
    // Step t >= 1: flips walked bit ctz(t); returns the walked bits' new state.
    __device__ __forceinline__ unsigned step(const RoiShared<L>& s, unsigned t) {
        const int b = __builtin_ctz(t) + kRoiGroupBits;
        const unsigned gray = t ^ (t >> 1);
        const bool on = (gray >> (b - kRoiGroupBits)) & 1u;   // after the flip
        const double d = on ? 1.0 : -1.0;
        double fb = 0.0;
#pragma unroll
        for (int j = kRoiGroupBits; j < L; ++j) fb = j == b ? f[j] : fb;
        e = fma(fb, d, e);   // d = +-1: the products are exact
        const double* row = s.J[b];
#pragma unroll
        for (int j = 0; j < L; ++j) f[j] = fma(row[j], d, f[j]);
        return gray;
    }
    // The group's energies.
    __device__ __forceinline__ void energies(const RoiShared<L>& s, double (&E)[kRoiStates]) const {
        E[0] = e;
#pragma unroll
        for (int a = 0; a < kRoiGroupBits; ++a) {
            double g[kRoiStates / 2];
            g[0] = f[a];
#pragma unroll
            for (int k = 0; k < a; ++k)
#pragma unroll
                for (int q = 0; q < (1 << k); ++q) g[(1 << k) + q] = g[q] + s.J[a][k];
#pragma unroll
            for (int q = 0; q < (1 << a); ++q) E[(1 << a) + q] = E[q] + g[q];
        }
    }
};

}  // namespace

// Every block's minimum energy and the smallest state index that has it.
template <int B>
__global__ void __launch_bounds__(kRoiBlock) roi_min_kernel(int n, const double* h, const double* Js, double* blk_e,
                                                            uint64_t* blk_s) {
    constexpr int L = kRoiGroupBits + B;
    __shared__ RoiShared<L> s;
    __shared__ double re[kRoiBlock];
    __shared__ uint64_t rs[kRoiBlock];
    roi_stage<L>(n, h, Js, blockIdx.x, s);
    RoiWalk<B> w;
    w.start(s);
    double best = __builtin_huge_val();
    unsigned best_g = 0;
    RoiWalk<B> at = w;   // the walk at the best group
#pragma unroll 1
    for (unsigned t = 0; t < (1u << B); ++t) {
        const unsigned gray = t > 0 ? w.step(s, t) : 0u;
        double E[kRoiStates];
        w.energies(s, E);
#pragma unroll
        for (int m = kRoiStates / 2; m > 0; m >>= 1)
#pragma unroll
            for (int q = 0; q < m; ++q) E[q] = fmin(E[q], E[q + m]);
        if (E[0] < best || (E[0] == best && gray < best_g)) {
            best = E[0];
            best_g = gray;
            at.e = w.e;
#pragma unroll
            for (int a = 0; a < kRoiGroupBits; ++a) at.f[a] = w.f[a];
        }
    }
    // the smallest of the best group's states at that energy
    double E[kRoiStates];
    at.energies(s, E);
    unsigned low = 0;
#pragma unroll
    for (int q = kRoiStates - 1; q >= 0; --q) low = E[q] == best ? unsigned(q) : low;
    re[threadIdx.x] = best;
    rs[threadIdx.x] = (uint64_t(blockIdx.x) << (L + kRoiThreadBits)) | (uint64_t(threadIdx.x) << L) |
                      (uint64_t(best_g) << kRoiGroupBits) | low;
    __syncthreads();
    for (int w2 = kRoiBlock / 2; w2 > 0; w2 /= 2) {
        if (int(threadIdx.x) < w2) {
            const double eo = re[threadIdx.x + w2];
            const uint64_t so = rs[threadIdx.x + w2];
            if (eo < re[threadIdx.x] || (eo == re[threadIdx.x] && so < rs[threadIdx.x])) {
                re[threadIdx.x] = eo;
                rs[threadIdx.x] = so;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        blk_e[blockIdx.x] = re[0];
        blk_s[blockIdx.x] = rs[0];
    }
}

// The minimum over the blocks, one workgroup.
__global__ void __launch_bounds__(1024) roi_min_final_kernel(int blocks, const double* blk_e, const uint64_t* blk_s,
                                                             double* e_min, uint64_t* s_min) {
    __shared__ double re[1024];
    __shared__ uint64_t rs[1024];
    const int t = int(threadIdx.x);
    double e = __builtin_huge_val();
    uint64_t st = ~uint64_t(0);
    for (int b = t; b < blocks; b += 1024)
        if (blk_e[b] < e || (blk_e[b] == e && blk_s[b] < st)) {
            e = blk_e[b];
            st = blk_s[b];
        }
    re[t] = e;
    rs[t] = st;
    __syncthreads();
    for (int w = 512; w > 0; w /= 2) {
        if (t < w && (re[t + w] < re[t] || (re[t + w] == re[t] && rs[t + w] < rs[t]))) {
            re[t] = re[t + w];
            rs[t] = rs[t + w];
        }
        __syncthreads();
    }
    if (t == 0) {
        *e_min = re[0];
        *s_min = rs[0];
    }
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Z and the weighted sums of the low and thread bits of every block (kRoiSums values: Z, the
// low bits', the thread bits'). PROD: a group's weights as products of 6 exponentials --
// made and summed relative to its first state's, which the host's check holds between e^-600
// and e^600, so none of them leaves a double's ordinary range; each sum is then scaled by the
// first state's weight, in two factors of its root, as that weight itself may underflow where
// the group's other states have weights a marginal is made of. A sum thus keeps its accuracy
// down to a double's smallest ordinary value, as one exponential per state does (the other form).
// The scaling is 12 multiplications in about 320 instructions a group (a call: 26 bits 0.133 ms, 32
// bits 2.13 ms, both as without it).
template <int B, bool PROD>
__global__ void __launch_bounds__(kRoiBlock) roi_sum_kernel(int n, const double* h, const double* Js, double beta,
                                                            const double* e_min, const double* factors, double* blk) {
    constexpr int L = kRoiGroupBits + B;
    constexpr int kWaves = kRoiBlock / 64;
    __shared__ RoiShared<L> s;
    __shared__ double red[kWaves][kRoiSums];
    roi_stage<L>(n, h, Js, blockIdx.x, s);
    const double e_ref = *e_min;
    RoiWalk<B> w;
    w.start(s);
    double z = 0.0, m[L];
#pragma unroll
    for (int j = 0; j < L; ++j) m[j] = 0.0;
#pragma unroll 1
    for (unsigned t = 0; t < (1u << B); ++t) {
        const unsigned gray = t > 0 ? w.step(s, t) : 0u;
        double W[kRoiStates];
        if constexpr (PROD) {
            W[0] = 1.0;
#pragma unroll
            for (int a = 0; a < kRoiGroupBits; ++a) {
                double T[kRoiStates / 2];
                T[0] = exp(-beta * w.f[a]);
#pragma unroll
                for (int k = 0; k < a; ++k)
#pragma unroll
                    for (int q = 0; q < (1 << k); ++q) T[(1 << k) + q] = T[q] * factors[a * kRoiGroupBits + k];
#pragma unroll
                for (int q = 0; q < (1 << a); ++q) W[(1 << a) + q] = W[q] * T[q];
            }
        } else {
            w.energies(s, W);
#pragma unroll
            for (int q = 0; q < kRoiStates; ++q) W[q] = exp(-beta * (W[q] - e_ref));
        }
        const double root = PROD ? exp(-0.5 * beta * (w.e - e_ref)) : 1.0;
        auto scaled = [&](double v) { return PROD ? v * root * root : v; };
        // pairwise over the group's bits: the odd half of each level is that bit's weight
#pragma unroll
        for (int a = 0; a < kRoiGroupBits; ++a) {
            constexpr int kHalf = kRoiStates / 2;
            const int half = kHalf >> a;
            double odd = 0.0;
#pragma unroll
            for (int q = 0; q < kHalf; ++q)
                if (q < half) {
                    odd += W[2 * q + 1];
                    W[q] = W[2 * q] + W[2 * q + 1];
                }
            m[a] += scaled(odd);
        }
        const double zg = scaled(W[0]);
        z += zg;
#pragma unroll
        for (int j = kRoiGroupBits; j < L; ++j) m[j] += ((gray >> (j - kRoiGroupBits)) & 1u) ? zg : 0.0;
    }
    const int lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
    auto put = [&](int k, double v) {
        v = wave_sum(v);
        if (lane == 0) red[wave][k] = v;
    };
    put(0, z);
#pragma unroll
    for (int j = 0; j < L; ++j) put(1 + j, m[j]);
#pragma unroll
    for (int t = 0; t < kRoiThreadBits; ++t) put(1 + L + t, ((threadIdx.x >> t) & 1u) ? z : 0.0);
    __syncthreads();
    if (int(threadIdx.x) < 1 + L + kRoiThreadBits) {
        double v = red[0][threadIdx.x];
        for (int q = 1; q < kWaves; ++q) v += red[q][threadIdx.x];
        blk[size_t(blockIdx.x) * kRoiSums + threadIdx.x] = v;
    }
}

// Value k over the blocks (0: Z, 1 + i: bit i's weight): the blocks' own sums for the low and
// thread bits, the Z of the blocks that have the bit set for a block bit. One workgroup per
// value.
__global__ void __launch_bounds__(256) roi_sum_final_kernel(int blocks, int low, const double* blk, double* out) {
    __shared__ double red[256];
    const int k = int(blockIdx.x), t = int(threadIdx.x);
    const int block_bit = k - 1 - (low + kRoiThreadBits);   // >= 0: a block bit
    double v = 0.0;
    for (int b = t; b < blocks; b += 256) {
        if (block_bit >= 0) v += ((b >> block_bit) & 1) ? blk[size_t(b) * kRoiSums] : 0.0;
        else v += blk[size_t(b) * kRoiSums + k];
    }
    red[t] = v;
    __syncthreads();
    for (int w = 128; w > 0; w /= 2) {
        if (t < w) red[t] += red[t + w];
        __syncthreads();
    }
    if (t == 0) out[k] = red[0];
}

// Walked bits at n bits: enough threads for 16 waves per CU first, then longer walks.
int roi_walked_bits(int n) {
    const int b = n - kRoiGroupBits - 18;
    return b < 0 ? 0 : (b > kRoiMaxWalked ? kRoiMaxWalked : b);
}

template <typename F>
static hipError_t with_walked(int b, F&& fn) {
    static_assert(kRoiMaxWalked == 7, "one case per walk length");
    switch (b) {
        case 0: return fn.template operator()<0>();
        case 1: return fn.template operator()<1>();
        case 2: return fn.template operator()<2>();
        case 3: return fn.template operator()<3>();
        case 4: return fn.template operator()<4>();
        case 5: return fn.template operator()<5>();
        case 6: return fn.template operator()<6>();
        case 7: return fn.template operator()<7>();
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_roi_min(int n, const double* h, const double* Js, double* blk_e, uint64_t* blk_s, double* e_min,
                          uint64_t* s_min, hipStream_t st) {
    const unsigned blocks = roi_blocks(n);
    const hipError_t e = with_walked(roi_walked_bits(n), [&]<int B>() {
        roi_min_kernel<B><<<blocks, kRoiBlock, 0, st>>>(n, h, Js, blk_e, blk_s);
        return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    roi_min_final_kernel<<<1, 1024, 0, st>>>(int(blocks), blk_e, blk_s, e_min, s_min);
    return hipGetLastError();
}

hipError_t launch_roi_sum(int n, const double* h, const double* Js, double beta, const double* e_min,
                          const double* factors, bool products, double* blk, double* out, hipStream_t st) {
    const unsigned blocks = roi_blocks(n);
    const int b = roi_walked_bits(n);
    const hipError_t e = with_walked(b, [&]<int B>() {
        if (products) roi_sum_kernel<B, true><<<blocks, kRoiBlock, 0, st>>>(n, h, Js, beta, e_min, factors, blk);
        else roi_sum_kernel<B, false><<<blocks, kRoiBlock, 0, st>>>(n, h, Js, beta, e_min, factors, blk);
        return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    roi_sum_final_kernel<<<unsigned(n + 1), 256, 0, st>>>(int(blocks), kRoiGroupBits + b, blk, out);
    return hipGetLastError();
}

}  // namespace qb
