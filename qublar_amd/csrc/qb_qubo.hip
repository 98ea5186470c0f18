// qb_qubo.hip -- gfx950 kernels of the batched sparse-QUBO engine.
//
// A batch holds many independent QUBOs, E(x) = sum_i h_i x_i + sum_{i<j} J_ij x_i x_j
// over x in {0,1}^n, each with its own replicas. The work unit is a job: one instance
// and a block of RB of its replicas. Jobs share nothing, so the persistent kernel takes
// them from queues with no inter-workgroup synchronisation, and a workgroup anneals its
// job alone. Each instance belongs to one XCD's queue (instances spread over the eight
// by decreasing cost), its jobs side by side, so the jobs of an instance run together on
// one XCD and read its rows through that XCD's L2; a workgroup whose queue is empty takes
// from the others. Inside a job: every sweep visits the instance's colour classes in
// order, a class is a set of independent flips, and the workgroup syncs between classes.
//
// Inside a class each lane takes one bit for all the job's replicas: it walks the bit's
// row once (walk_row) and adds each coupling into the accumulator of every replica whose
// neighbour spin is set -- in row order, per replica.
// The spin words of a job (bit r of word i = replica r0 + r's x_i) live in the
// workgroup's LDS while it anneals (global memory only for instances too large for it),
// so the random reads of neighbours' spins never leave the CU.
//
// dE of flipping bit i = (1 - 2 x_i)(h_i + sum_j J_ij x_j), summed in FP64 in CSR order,
// and a flip is accepted iff dE <= 0 or u < qexp(-dE * beta) -- the ray x voxel engine's
// test, decided through a float exponential with a guard band (uphill_accept). Replicas 2m and 2m + 1 share one Philox4x32-10 call keyed by the instance seed with
// counter (bit, sweep, m, tag), one 53-bit uniform each (draw2_u01).
#include <algorithm>

#include "qb_internal.h"
#include "qb_rng.h"

namespace qb {

// Spin words of a job in LDS: one byte per bit up to 8 replicas per job, 16 or 32 bits
// beyond; kQuboLdsBytes of them hold instances up to kQuboLdsBytes / sizeof(word) bits.
template <int RB>
struct LdsWord {
    using type = uint32_t;
};
template <>
struct LdsWord<4> {
    using type = uint8_t;
};
template <>
struct LdsWord<8> {
    using type = uint8_t;
};
template <>
struct LdsWord<16> {
    using type = uint16_t;
};

// Bits a spin word is shifted up by: four replicas to a byte lie in its upper half, where
// walk_row wants them.
template <int RB, typename W>
constexpr int word_shift() {
    return RB <= 4 && sizeof(W) == 1 ? 4 : 0;
}

// N entries of a tile's rows: columns and couplings, then the neighbours' spin words, all in
// flight together; each coupling goes into the accumulator of every replica whose neighbour
// spin is set, in row order, as fma(w, x_j, acc): w x_j is exact, so each addition rounds once
// as acc + w does, and an unset neighbour -- or a padding entry, whose coupling is zero --
// leaves acc (up to the sign of an exact zero, which no decision sees).
//
// The sums are most of a sweep's instructions. With four replicas to a byte, a
// multiplication spreads the nibble to one bit a byte and each replica's x_j, as 0 or 2.0, is
// one byte moved to the top of a double: two instructions per (entry, replica) where bit
// field, conversion and FMA are three (the accumulators hold twice the sums). Rows padded to
// their tile's longest need no test per entry, and a tile's steps are its own length (16, then
// 8, 4, 2 and 1 entries), not whole steps of 16. 48 instances of 1,000 to 16,384 bits, degrees
// 3 to 64, 8 to 32 replicas, 400 sweeps: 86.5 -> 53.7 ms. (x_j as any one exponent bit of a
// double would save the moved byte too, but factors of 2^-511 and below slow the FMAs: 280.) There,
// with the long jobs halved, a CU with a job has a vector instruction in 47% of its SIMDs' cycles
// and its LDS active in 18%, its waves waiting for the rows' and spins' loads in between; a CU
// has a job 42% of the time.
template <int RB, int N, int SHIFT, typename W>
__device__ __forceinline__ void walk_row(const int* tcol, const float* tJ, const W* mk, double (&acc)[RB]) {
    const unsigned lane = threadIdx.x % 64;
    int cj[N];
    float wj[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
        cj[u] = tcol[lane + 64u * u];
        wj[u] = tJ[lane + 64u * u];
    }
    uint32_t mj[N];
#pragma unroll
    for (int u = 0; u < N; ++u) mj[u] = uint32_t(mk[cj[u]]);
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const double w = double(wj[u]);
        if constexpr (SHIFT != 0) {
            static_assert(RB <= 4 && SHIFT == 4);
            const uint32_t word = (mj[u] * 0x810204u) & 0x40404040u;   // bit 4 + r to bit 8 r + 6
#pragma unroll
            for (int r = 0; r < RB; ++r) {
                const uint32_t hi = __builtin_amdgcn_perm(word, word, (uint32_t(r) << 24) | 0x0C0C0Cu);
                acc[r] = fma(w, __hiloint2double(int(hi), 0), acc[r]);
            }
        } else {
#pragma unroll
            for (int r = 0; r < RB; ++r) acc[r] = fma(w, double((mj[u] >> r) & 1u), acc[r]);
        }
    }
}

// One job's sweeps with its spin words at `mk` (LDS or global), local position index.
template <int RB, int BLOCK, typename W>
__device__ __forceinline__ void qubo_job(const DevQuboBatch& q, const QuboJob& jb, W* mk, const double* beta,
                                         int n_sweeps) {
    const int k = jb.instance, rb = jb.replicas;
    const int bit0 = q.inst_pos[k];
    const int c0 = q.inst_cls[k], c1 = q.inst_cls[k + 1];
    const uint64_t key = q.seed[k];
    const uint32_t pair0 = uint32_t(jb.replica0) / 2u;   // replica0 is a multiple of RB
    constexpr int kShift = word_shift<RB, W>();
    constexpr double kUnit = kShift ? 2.0 : 1.0;
    for (int sweep = 0; sweep < n_sweeps; ++sweep) {
        const double b = beta[sweep];
        for (int c = c0; c + 1 < c1; ++c) {
            const int lo = q.cls_ptr[c], hi = q.cls_ptr[c + 1];
            for (int pos = lo + int(threadIdx.x); pos < hi; pos += BLOCK) {
                const uint32_t mi = uint32_t(mk[pos - bit0]) >> kShift;
                const double hp = double(q.h[pos]) * kUnit;
                double acc[RB];
#pragma unroll
                for (int r = 0; r < RB; ++r) acc[r] = hp;
                const int tile = q.class_tile[c] + __builtin_amdgcn_readfirstlane((pos - lo) >> 6);
                const int at = q.tile_ptr[tile], end = q.tile_ptr[tile + 1];
                int e = at;
                for (; end - e >= 64 * 16; e += 64 * 16) walk_row<RB, 16, kShift>(q.tcol + e, q.tJ + e, mk, acc);
                if (end - e >= 64 * 8) {
                    walk_row<RB, 8, kShift>(q.tcol + e, q.tJ + e, mk, acc);
                    e += 64 * 8;
                }
                if (end - e >= 64 * 4) {
                    walk_row<RB, 4, kShift>(q.tcol + e, q.tJ + e, mk, acc);
                    e += 64 * 4;
                }
                if (end - e >= 64 * 2) {
                    walk_row<RB, 2, kShift>(q.tcol + e, q.tJ + e, mk, acc);
                    e += 64 * 2;
                }
                if (end - e >= 64) walk_row<RB, 1, kShift>(q.tcol + e, q.tJ + e, mk, acc);
                if constexpr (kShift != 0) {
#pragma unroll
                    for (int r = 0; r < RB; ++r) acc[r] *= 1.0 / kUnit;
                }
                const uint32_t bit = uint32_t(q.bit_id[pos]);
                uint32_t flips = 0;
#pragma unroll
                for (int r = 0; r < RB; r += 2) {
                    if (r < rb) {
                        double u[2];
                        draw2_u01(key, uint32_t(sweep), bit, pair0 + uint32_t(r / 2), u[0], u[1]);
#pragma unroll
                        for (int v = 0; v < 2; ++v) {
                            const double dE = ((mi >> (r + v)) & 1u) ? -acc[r + v] : acc[r + v];
                            if (r + v < rb && (dE <= 0.0 || uphill_accept(-dE * b, u[v]))) flips |= 1u << (r + v);
                        }
                    }
                }
                if (flips) mk[pos - bit0] = W((mi ^ flips) << kShift);
            }
            __syncthreads();
        }
    }
}

// The next job for this workgroup: from its own XCD's queue, else from the others in turn
// (a queue already read as exhausted costs no atomic); -1 when every queue is empty.
__device__ __forceinline__ int take_job(unsigned* queue, const QuboQueues& segs, int home) {
    for (int t = 0; t < kXcds; ++t) {
        const int x = (home + t) % kXcds;
        const int len = segs.begin[x + 1] - segs.begin[x];
        unsigned* ctr = queue + kQueueStride * x;
        if (len <= 0 || __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= unsigned(len)) continue;
        const unsigned k = atomicAdd(ctr, 1u);
        if (k < unsigned(len)) return segs.begin[x] + int(k);
    }
    return -1;
}

template <int RB, int BLOCK>
__global__ void __launch_bounds__(BLOCK) qubo_batch_kernel(DevQuboBatch q, uint32_t* masks, const double* beta,
                                                            int n_sweeps, unsigned* queue, QuboQueues segs) {
    static_assert(RB % 2 == 0, "replicas are drawn in pairs");
    using W = typename LdsWord<RB>::type;
    constexpr int kLdsBits = kQuboLdsBytes / int(sizeof(W));
    __shared__ W lmask[kLdsBits];
    __shared__ int s_job;
    const int home = int(xcc_id() % kXcds);
    for (;;) {
        if (threadIdx.x == 0) s_job = take_job(queue, segs, home);
        __syncthreads();
        const int jn = s_job;
        __syncthreads();   // s_job is written again by the next take
        if (jn < 0) return;
        const QuboJob jb = q.jobs[jn];
        const int n = q.inst_pos[jb.instance + 1] - q.inst_pos[jb.instance];
        uint32_t* gm = masks + jb.mask_offset;
        if (n <= kLdsBits) {
            // the job's spins live in LDS from all-zero x; written out once at the end
            for (int i = int(threadIdx.x); i < n; i += BLOCK) lmask[i] = W(0);
            __syncthreads();
            if (RB == 4 && jb.replicas <= 2) qubo_job<2, BLOCK, W>(q, jb, lmask, beta, n_sweeps);
            else qubo_job<RB, BLOCK, W>(q, jb, lmask, beta, n_sweeps);
            for (int i = int(threadIdx.x); i < n; i += BLOCK) gm[i] = uint32_t(lmask[i]) >> word_shift<RB, W>();
            __syncthreads();
        } else {
            qubo_job<RB, BLOCK, uint32_t>(q, jb, gm, beta, n_sweeps);
        }
    }
}

// FP64 energy of the replicas of every job, four of them per workgroup: a wave takes every
// 16th tile of the instance, a lane a bit of it for the four replicas, so a row is read once
// for all of them in whole lines, eight entries in flight; then a tree over the lanes and the
// waves. Bound by the latency of the spin words' gathers. 48 instances of 1,000 to 16,384
// bits, 8 to 32 replicas: 0.36 ms, where a workgroup per job that walked its replicas one
// after the other, a row per lane, took 5.6.
__global__ void __launch_bounds__(kQuboEnergyBlock) qubo_energy_kernel(DevQuboBatch q, const uint32_t* masks,
                                                                       double* energy) {
    constexpr int kR = 4, kFlight = 8, kWaves = kQuboEnergyBlock / 64;
    __shared__ double part[kR][kWaves];
    const QuboJob jb = q.jobs[blockIdx.x];
    const int r0 = int(blockIdx.y) * kR;
    if (r0 >= jb.replicas) return;   // the whole workgroup leaves
    const int k = jb.instance, lane = int(threadIdx.x) % 64;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / 64);
    const uint32_t* mk = masks + jb.mask_offset;
    const int bit0 = q.inst_pos[k];
    const int t1 = q.class_tile[q.inst_cls[k + 1] - 1];
    double e[kR] = {};
    for (int t = q.class_tile[q.inst_cls[k]] + wave; t < t1; t += kWaves) {
        const int pos = q.tile_pos[t] + lane;
        const bool valid = pos < q.tile_pos[t + 1];
        const uint32_t mi = valid ? mk[pos - bit0] >> r0 : 0u;
        double pair[kR] = {};
        // unsigned: the last step of rows that end at the int32 limit runs past it
        const unsigned at = unsigned(q.tile_ptr[t]), end = unsigned(q.tile_ptr[t + 1]);
        for (unsigned i = at; i < end; i += 64 * kFlight) {
            int cj[kFlight];
            float wj[kFlight];
            uint32_t mj[kFlight];
#pragma unroll
            for (int u = 0; u < kFlight; ++u) {
                const unsigned from = min(i + 64u * u, end - 64u) + unsigned(lane);
                cj[u] = q.tcol[from];
                wj[u] = q.tJ[from];
            }
#pragma unroll
            for (int u = 0; u < kFlight; ++u) mj[u] = i + 64u * u < end ? mk[cj[u]] >> r0 : 0u;
#pragma unroll
            for (int u = 0; u < kFlight; ++u)
#pragma unroll
                for (int r = 0; r < kR; ++r) pair[r] = fma(double(wj[u]), double((mj[u] >> r) & 1u), pair[r]);
        }
        const double h = valid ? double(q.h[pos]) : 0.0;
#pragma unroll
        for (int r = 0; r < kR; ++r)
            if ((mi >> r) & 1u) e[r] += h + 0.5 * pair[r];
    }
#pragma unroll
    for (int r = 0; r < kR; ++r) {
#pragma unroll
        for (int d = 32; d > 0; d /= 2) e[r] += __shfl_down(e[r], unsigned(d));
        if (lane == 0) part[r][wave] = e[r];
    }
    __syncthreads();
    const int r = int(threadIdx.x) / kWaves, w = int(threadIdx.x) % kWaves;   // 16 lanes a replica
    if (int(threadIdx.x) < kR * kWaves) {
        double v = part[r][w];
#pragma unroll
        for (int d = kWaves / 2; d > 0; d /= 2) v += __shfl_down(v, unsigned(d), kWaves);
        if (w == 0 && r0 + r < jb.replicas) energy[jb.energy_offset + r0 + r] = v;
    }
}

template <int BLOCK>
static hipError_t launch_qubo_block(const DevQuboBatch& q, int rb, uint32_t* masks, const double* beta, int n_sweeps,
                                    unsigned* queue, const QuboQueues& segs, int workgroups, hipStream_t st) {
    switch (rb) {
        case 4: qubo_batch_kernel<4, BLOCK><<<workgroups, BLOCK, 0, st>>>(q, masks, beta, n_sweeps, queue, segs); break;
        case 8: qubo_batch_kernel<8, BLOCK><<<workgroups, BLOCK, 0, st>>>(q, masks, beta, n_sweeps, queue, segs); break;
        case 16: qubo_batch_kernel<16, BLOCK><<<workgroups, BLOCK, 0, st>>>(q, masks, beta, n_sweeps, queue, segs); break;
        case 32: qubo_batch_kernel<32, BLOCK><<<workgroups, BLOCK, 0, st>>>(q, masks, beta, n_sweeps, queue, segs); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_qubo_batch(const DevQuboBatch& q, int rb, int block, uint32_t* masks, const double* beta,
                             int n_sweeps, unsigned* queue, const QuboQueues& segs, int workgroups, hipStream_t st) {
    for (int x = 0; x < kXcds; ++x)
        if (segs.begin[x] < 0 || segs.begin[x + 1] < segs.begin[x] || segs.begin[x + 1] > q.n_jobs)
            return hipErrorInvalidValue;
    if (block == 256) return launch_qubo_block<256>(q, rb, masks, beta, n_sweeps, queue, segs, workgroups, st);
    if (block == 1024) return launch_qubo_block<1024>(q, rb, masks, beta, n_sweeps, queue, segs, workgroups, st);
    return hipErrorInvalidValue;
}

int qubo_blocks_per_cu(int rb, int block) {
    int per_cu = 0;
    const void* k = nullptr;
    if (block == 256)
        k = rb == 4 ? (const void*)&qubo_batch_kernel<4, 256> : rb == 8 ? (const void*)&qubo_batch_kernel<8, 256>
          : rb == 16 ? (const void*)&qubo_batch_kernel<16, 256> : (const void*)&qubo_batch_kernel<32, 256>;
    else
        k = rb == 4 ? (const void*)&qubo_batch_kernel<4, 1024> : rb == 8 ? (const void*)&qubo_batch_kernel<8, 1024>
          : rb == 16 ? (const void*)&qubo_batch_kernel<16, 1024> : (const void*)&qubo_batch_kernel<32, 1024>;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, block, 0) != hipSuccess) return 0;
    return per_cu;
}

// A fill kernel in place of a memset where the launch schedule is recorded into a graph.
__global__ void fill_u32_kernel(uint32_t* p, size_t n, uint32_t v) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x) p[i] = v;
}

hipError_t launch_fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t st) {
    if (n == 0) return hipSuccess;
    const size_t blocks = std::min<size_t>((n + 255) / 256, 4096);
    fill_u32_kernel<<<unsigned(blocks), 256, 0, st>>>(p, n, v);
    return hipGetLastError();
}

hipError_t launch_qubo_energy(const DevQuboBatch& q, int rb, const uint32_t* masks, double* energy, hipStream_t st) {
    qubo_energy_kernel<<<dim3(unsigned(q.n_jobs), unsigned((rb + 3) / 4)), kQuboEnergyBlock, 0, st>>>(q, masks, energy);
    return hipGetLastError();
}

}  // namespace qb
