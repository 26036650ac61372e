// gfx950 FP32 CQ GEMV for batches of two or more activation rows:
//   y[b][row] = sum_g half(norm[row][g]) * (((0 + cb[c0] x0) + cb[c1] x1) + ...)
// in the reference's order, every product and every sum rounded on its own
// (cq.cpp:104-107, 157-164, 185-194), so outputs are bit-identical to the
// one-row kernels of cq_kernels.hip.
//
// What bounds it: the sequential fp32 sums, one v_add per (code, batch row).
// The one-row kernels look every product up in an LDS table (one LDS read,
// one offset op and one add per code and batch row, tables rebuilt per batch
// row). Here a code is looked up once for all batch rows, as its fp32
// centroid, and the matrix cores form the products:
// v_mfma_f32_4x4x1_16b_f32 with C = 0 has K = 1, so each output is one
// product rounded to fp32 (denormals included; an underflow to -0 stays -0,
// which no later sum can tell from +0). Operand A holds four batch rows x 16
// positions in one register; cbsz = 4 broadcasts the block that abid names,
// so the four rows' values of position 16-block/abid reach every lane
// without a move. Operand B is the centroid of lane l's weight row, and
// output register i of lane l is row l's product with batch row i: the add
// chains stay in the weight row's lane. Per code: one MFMA per four batch
// rows, one add per batch row, and 1 (4-bit) or 0.5 (2-bit) offset ops and
// LDS reads in all. 8 adds + 2 MFMAs measured 16.3-17.4 ns per position and
// SIMD with 4 or 2 waves (10 issue slots of 4 clocks; 27.7 ns with one wave),
// so the launch aims at two waves per SIMD or more. Measured with the transform
// pre-pass: 16 x CQ2 4096 x 4096 g128 at 8 rows 191 -> 100 us (one row per pass
// before), 16 x CQ4 8192 x 8192 g32 at 4 / 8 / 16 rows 402 / 742 / 1428 -> 287 /
// 473 / 813 us (rows in pairs before).
#pragma once

#include "batch_pick.h"
#include "codes.h"
#include "common.h"
#include "wave.h"

#include <hip/hip_fp16.h>

#include <type_traits>
#include <utility>

namespace nd {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kBlock = 64;  // positions handled between two rounds of loads

template <int KIND, int GROUP, int NB>
struct BatchShape {
    static constexpr int kQuads = (NB + 3) / 4;                    // operand registers of four batch rows
    static constexpr int kCodesPerDword = KIND == kNib ? 8 : 16;
    static constexpr int kDwords = kBlock / kCodesPerDword;        // code dwords per block: 8 or 4
    static constexpr int kChunks = kDwords / 4;                    // 16-byte chunks per block: 2 or 1
    static constexpr int kNorms = GROUP < kBlock ? kBlock / GROUP : 1;
};

template <int KIND, int GROUP, int NB>
struct BatchState {
    using S = BatchShape<KIND, GROUP, NB>;
    u32x4 codes[S::kChunks];
    f4 x[S::kQuads];  // lane l: batch row l % 4 of the quad, positions 4 (l / 4) .. + 4 of the block
    uint16_t norms[S::kNorms];
};

struct BatchPtrs {
    __amdgpu_buffer_rsrc_t codes, norms, x;
    uint32_t code_lane, norm_lane;
    int bpg_shift;  // log2(blocks per group), 0 for groups of at most a block
};

template <int KIND, int GROUP, int NB>
__device__ __forceinline__ u32x4 batch_chunk(const BatchPtrs &p, int block, int c) {
    constexpr int C = BatchShape<KIND, GROUP, NB>::kChunks;
    return __builtin_amdgcn_raw_buffer_load_b128(
        p.codes, p.code_lane, __builtin_amdgcn_readfirstlane((block * C + c) * kRowsPerBlock * 16), kStreamLoad);
}

// The block's group norms (a group past the last reads zero and is never added).
template <int KIND, int GROUP, int NB>
__device__ __forceinline__ void batch_norms(BatchState<KIND, GROUP, NB> &st, const BatchPtrs &p, int block) {
    constexpr int NN = BatchShape<KIND, GROUP, NB>::kNorms;
#pragma unroll
    for (int k = 0; k < NN; ++k) {
        const int g = GROUP < kBlock ? block * NN + k : block >> p.bpg_shift;
        st.norms[k] = __builtin_amdgcn_raw_buffer_load_b16(
            p.norms, p.norm_lane, __builtin_amdgcn_readfirstlane(g * kRowsPerBlock * 2), 0);
    }
}

// The block's activations. XF: from the raw rows (zeros past the row's end,
// the reference's padding), then the group FWHT in registers with the
// reference's stage order and operands: position 4 (l / 4) + e, so strides 1
// and 2 pair the lane's own values and stride h >= 4 pairs lanes l and l ^ h.
template <int KIND, int GROUP, int NB, bool XF>
__device__ __forceinline__ void batch_x(BatchState<KIND, GROUP, NB> &st, const BatchPtrs &p,
                                        const uint32_t (&xv)[BatchShape<KIND, GROUP, NB>::kQuads], int block, int in) {
    const int so = __builtin_amdgcn_readfirstlane(block * kBlock * 4);
#pragma unroll
    for (int q = 0; q < BatchShape<KIND, GROUP, NB>::kQuads; ++q) {
        if constexpr (!XF) {
            st.x[q] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(p.x, xv[q], so, 0));
        } else {
            const int p0 = block * kBlock + 4 * ((threadIdx.x & 63) >> 2);
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // an offset past the resource reads zero
                const uint32_t off = p0 + e < in ? xv[q] + 4u * e + so : 0xFFFFFFF0u;
                v[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(p.x, off, 0, 0));
            }
            st.x[q] = f4{v[0], v[1], v[2], v[3]};
        }
    }
}

template <int KIND, int GROUP, int NB, bool XF>
__device__ __forceinline__ void batch_transform(BatchState<KIND, GROUP, NB> &st, float scale) {
    if constexpr (XF) {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int q = 0; q < BatchShape<KIND, GROUP, NB>::kQuads; ++q) {
            float a = st.x[q].x + st.x[q].y, b = st.x[q].x - st.x[q].y;
            float c = st.x[q].z + st.x[q].w, d = st.x[q].z - st.x[q].w;
            float v[4] = {a + c, b + d, a - c, b - d};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                wave_butterflies<GROUP, 4>(v[e], lane);
                v[e] = v[e] * scale;
            }
            st.x[q] = f4{v[0], v[1], v[2], v[3]};
        }
    }
}

// Centroids of one code dword: lane l's row, 8 or 16 consecutive positions.
template <int KIND>
struct Centroids {
    float v[KIND == kNib ? 8 : 16];
};

template <int KIND>
__device__ __forceinline__ void read_centroids(Centroids<KIND> &w, const float *table, uint32_t dword, uint32_t mask) {
    uint32_t off[8];
    slot_offsets_sdwa<KIND>(dword, mask, off);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const char *e = reinterpret_cast<const char *>(table) + off[i];
        if constexpr (KIND == kNib) {
            w.v[i] = *reinterpret_cast<const float *>(e);
        } else {
            const float2 pr = *reinterpret_cast<const float2 *>(e);
            w.v[2 * i] = pr.x;
            w.v[2 * i + 1] = pr.y;
        }
    }
}

template <int Q>
struct Products {
    f4 v[Q];
};

// Products of position P of the block with every batch row of the tile.
template <int KIND, int GROUP, int NB, int P>
__device__ __forceinline__ void products(Products<BatchShape<KIND, GROUP, NB>::kQuads> &pr,
                                         const BatchState<KIND, GROUP, NB> &st, float w) {
#pragma unroll
    for (int q = 0; q < BatchShape<KIND, GROUP, NB>::kQuads; ++q)
        pr.v[q] = __builtin_amdgcn_mfma_f32_4x4x1f32(st.x[q][P & 3], w, f4{0.0f, 0.0f, 0.0f, 0.0f}, 4, P >> 2, 0);
}

template <int N, class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

// KS parts of 256 threads share a row tile, part k taking rounds k, KS + k,
// ... of max(64, GROUP) positions; parts above 0 park their group terms in
// LDS and part 0 adds them in group order, one round behind (the scheme of
// the quarter-split kernel in cq_kernels.hip).
template <int KIND, int GROUP, int NB, int KS>
struct ParkShape {
    static constexpr int kTerms = BatchShape<KIND, GROUP, NB>::kNorms * NB;  // per part, round and row
    static constexpr int kFloats = KS > 1 ? (KS - 1) * kTerms * kRowsPerBlock : 1;
    static constexpr int kBuffers = KS > 1 ? 2 : 1;
};

template <int KIND, int GROUP, int NB, int KS, bool XF, bool FIRST>
__device__ __forceinline__ void batch_rows(const CqJob &J, const CqGeom &geom, const float *table,
                                           float (*park)[ParkShape<KIND, GROUP, NB, KS>::kFloats], int blk, int b0,
                                           int part) {
    using S = BatchShape<KIND, GROUP, NB>;
    constexpr int NN = S::kNorms, NQ = S::kQuads, D = S::kDwords, CPD = S::kCodesPerDword;
    const int r = threadIdx.x % kRowsPerBlock, lane = threadIdx.x & 63;
    const int tile = blk - J.block_begin;
    const int nb = min(NB, J.batch - b0);
    const int stride = XF ? geom.in : geom.windows * kWindow;
    BatchPtrs p;
    p.codes = buffer_rsrc(J.codes + static_cast<size_t>(tile) * geom.chunks * kRowsPerBlock,
                          static_cast<uint32_t>(geom.chunks) * kRowsPerBlock * 16u);
    p.norms = buffer_rsrc(J.norms + static_cast<size_t>(tile) * geom.groups * kRowsPerBlock,
                          static_cast<uint32_t>(geom.groups) * kRowsPerBlock * 2u);
    p.x = buffer_rsrc(J.act + static_cast<size_t>(b0) * stride, static_cast<uint32_t>(nb) * stride * 4u);
    p.code_lane = r * 16u;
    p.norm_lane = r * 2u;
    p.bpg_shift = GROUP < kBlock ? 0 : __builtin_ctz(geom.group / kBlock);
    uint32_t xv[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q)  // rows past the batch repeat its last row; their outputs are not stored
        xv[q] = (static_cast<uint32_t>(min(4 * q + (lane & 3), nb - 1)) * stride + 4 * (lane >> 2)) * 4u;

    const int groups = geom.groups;
    const int bpg = 1 << p.bpg_shift;
    const int blocks = GROUP < kBlock ? (groups + NN - 1) / NN : groups << p.bpg_shift;
    const int rounds = (blocks + (KS << p.bpg_shift) - 1) / (KS << p.bpg_shift);
    const int count = rounds << p.bpg_shift;  // blocks this part walks (past the row's end: never added)
    // block n of this part
    auto block_of = [&](int n) { return (((n >> p.bpg_shift) * KS + part) << p.bpg_shift) + (n & (bpg - 1)); };

    BatchState<KIND, GROUP, NB> st[2];
    auto load = [&](BatchState<KIND, GROUP, NB> &s, int n) {
        const int block = block_of(n);
#pragma unroll
        for (int c = 0; c < S::kChunks; ++c) s.codes[c] = batch_chunk<KIND, GROUP, NB>(p, block, c);
        batch_x<KIND, GROUP, NB, XF>(s, p, xv, block, geom.in);
        batch_norms<KIND, GROUP, NB>(s, p, block);
    };
    load(st[0], 0);
    load(st[1], 1);
    const uint32_t mask = KIND == kNib ? 0x3Cu : 0x78u;
    float sum[NB], gd[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) sum[b] = 0.0f, gd[b] = 0.0f;
    Centroids<KIND> w[2];
    batch_transform<KIND, GROUP, NB, XF>(st[0], geom.scale);
    read_centroids<KIND>(w[0], table, st[0].codes[0].x, mask);

    // the parked terms of round `it`
    auto add_parked = [&](int it) {
        const float *src = park[it & 1] + r;
#pragma unroll
        for (int k = 1; k < KS; ++k)
#pragma unroll
            for (int j = 0; j < NN; ++j)
                if ((it * KS + k) * NN + j < groups)
#pragma unroll
                    for (int b = 0; b < NB; ++b) sum[b] += src[(((k - 1) * NN + j) * NB + b) * kRowsPerBlock];
    };
    auto close = [&](int it, int k, uint16_t norm) {
        const float nf = __half2float(__ushort_as_half(norm));
        if constexpr (FIRST) {
            if (it * KS * NN + k < groups)
#pragma unroll
                for (int b = 0; b < NB; ++b) sum[b] += gd[b] * nf;
        } else {
            float *dst = park[it & 1] + r;
#pragma unroll
            for (int b = 0; b < NB; ++b) dst[(((part - 1) * NN + k) * NB + b) * kRowsPerBlock] = gd[b] * nf;
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) gd[b] = 0.0f;
    };
    // One block: centroids are read one code dword ahead (the next block's
    // first dword during the last), products are formed one position ahead of
    // their adds, spent registers are refilled two blocks ahead.
    auto block_step = [&](auto slot, int n) {
        constexpr int cur = decltype(slot)::value;
        BatchState<KIND, GROUP, NB> &s = st[cur], &t = st[cur ^ 1];
        const int it = n >> p.bpg_shift;
        const int ahead = block_of(n + 2);
        if constexpr (FIRST && KS > 1) {
            if ((n & (bpg - 1)) == 0 && it > 0) add_parked(it - 1);
        }
        Products<NQ> pr[2];
        products<KIND, GROUP, NB, 0>(pr[0], s, w[0].v[0]);
        static_for<D>([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            constexpr int dn = d + 1;
            const u32x4 &cn = dn < D ? s.codes[dn / 4 % S::kChunks] : t.codes[0];
            constexpr int e = dn & 3;
            read_centroids<KIND>(w[dn & 1], table, e == 0 ? cn.x : e == 1 ? cn.y : e == 2 ? cn.z : cn.w, mask);
            if constexpr (e == 3 && dn < D) s.codes[dn / 4] = batch_chunk<KIND, GROUP, NB>(p, ahead, dn / 4);
            __builtin_amdgcn_sched_barrier(0);
            static_for<CPD>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                constexpr int P = d * CPD + i;
                if constexpr (P + 1 < kBlock)
                    products<KIND, GROUP, NB, (P + 1) % kBlock>(pr[(P + 1) & 1], s, w[(P + 1) / CPD & 1].v[(P + 1) % CPD]);
#pragma unroll
                for (int b = 0; b < NB; ++b) gd[b] += pr[P & 1].v[b / 4][b & 3];
                if constexpr (GROUP < kBlock && (P + 1) % GROUP == 0) close(it, (P + 1) / GROUP - 1, s.norms[(P + 1) / GROUP - 1]);
                // pins the position's adds and the next one's products here (they have no other order)
#pragma unroll
                for (int b = 0; b < NB; ++b) asm volatile("" : "+v"(gd[b]));
                if constexpr (P + 1 < kBlock) {
#pragma unroll
                    for (int q = 0; q < NQ; ++q) asm volatile("" : "+v"(pr[(P + 1) & 1].v[q]));
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        if constexpr (GROUP >= kBlock) {
            if ((n & (bpg - 1)) == bpg - 1) close(it, 0, s.norms[0]);
        }
        batch_x<KIND, GROUP, NB, XF>(s, p, xv, ahead, geom.in);
        batch_norms<KIND, GROUP, NB>(s, p, ahead);
        batch_transform<KIND, GROUP, NB, XF>(t, geom.scale);
        if constexpr (KS > 1) {
            if ((n & (bpg - 1)) == bpg - 1) __syncthreads();
        }
    };
    int n = 0;
    for (; n + 2 <= count; n += 2) {
        block_step(std::integral_constant<int, 0>{}, n);
        block_step(std::integral_constant<int, 1>{}, n + 1);
    }
    if (n < count) block_step(std::integral_constant<int, 0>{}, n);
    if constexpr (FIRST) {
        if constexpr (KS > 1) add_parked(rounds - 1);
        const int row = tile * kRowsPerBlock + r;
        const size_t ys = J.ystride ? J.ystride : J.rows;
        if (row < J.rows) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (b < nb) ((ND_GLOBAL float *)J.y)[static_cast<size_t>(b0 + b) * ys + row] = sum[b];
        }
    }
}

template <int KIND, int GROUP, int NB, int KS, bool XF>
__global__ __launch_bounds__(kRowsPerBlock *KS, 2) void cq_gemv_batch_kernel(CqJob job0, const CqJob *__restrict__ jobs,
                                                                           int njobs, int batch, CqGeom geom) {
    using PS = ParkShape<KIND, GROUP, NB, KS>;
    __shared__ __attribute__((aligned(16))) float table[KIND == kNib ? 16 : 32];
    __shared__ float park[PS::kBuffers][PS::kFloats];
    const int blk = blockIdx.x, b0 = blockIdx.y * NB;
    CqJob J = job0;
    if (njobs > 0) {
        const ND_CONST CqJob *cj = (const ND_CONST CqJob *)(jobs);
        const int j = find_job(cj, njobs, blk);
        J.codes = cj[j].codes;
        J.norms = cj[j].norms;
        J.act = cj[j].act;
        J.y = cj[j].y;
        J.rows = cj[j].rows;
        J.block_begin = cj[j].block_begin;
        J.ystride = cj[j].ystride;
    }
    J.batch = batch;
    // centroid of every code (4-bit), or the two centroids of every code pair (2-bit)
#pragma unroll
    for (int i = 0; i < (KIND == kNib ? 16 : 32); ++i)
        if (threadIdx.x == static_cast<unsigned>(i))
            table[i] = geom.lut[KIND == kNib ? i : (i & 1) ? i >> 3 : i >> 1 & 3];
    __syncthreads();
    const int part = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kRowsPerBlock) : 0;
    if (part == 0) batch_rows<KIND, GROUP, NB, KS, XF, true>(J, geom, table, park, blk, b0, 0);
    else batch_rows<KIND, GROUP, NB, KS, XF, KS == 1>(J, geom, table, park, blk, b0, part);
}

template <int KIND, int GROUP, int NB, int KS>
void launch_shape(const CqGeom &g, const CqJob &job0, const CqJob *jobs, int njobs, int blocks, int batch, bool x_raw,
                  hipStream_t s) {
    const dim3 grid(blocks, (batch + NB - 1) / NB), block(kRowsPerBlock * KS);
    if (x_raw) hipLaunchKernelGGL((cq_gemv_batch_kernel<KIND, GROUP, NB, KS, true>), grid, block, 0, s, job0, jobs, njobs, batch, g);
    else hipLaunchKernelGGL((cq_gemv_batch_kernel<KIND, GROUP, NB, KS, false>), grid, block, 0, s, job0, jobs, njobs, batch, g);
    ND_HIP(hipGetLastError());
}

template <int KIND, int GROUP, int NB>
void launch_parts(const CqGeom &g, const CqJob &job0, const CqJob *jobs, int njobs, int blocks, int batch, bool x_raw,
                  int ks, hipStream_t s) {
    if constexpr (GROUP >= 32) {
        if (ks == 4) return launch_shape<KIND, GROUP, NB, 4>(g, job0, jobs, njobs, blocks, batch, x_raw, s);
    }
    launch_shape<KIND, GROUP, NB, 1>(g, job0, jobs, njobs, blocks, batch, x_raw, s);
}

template <int KIND, int GROUP>
void launch_group(const CqGeom &g, const CqJob &job0, const CqJob *jobs, int njobs, int blocks, int batch, bool x_raw,
                  hipStream_t s) {
    const BatchPick b = batch_pick(g.kind, g.group, g.groups, blocks, batch);
    if constexpr (GROUP >= 32) {
        if (b.nb == 3) return launch_parts<KIND, GROUP, 3>(g, job0, jobs, njobs, blocks, batch, x_raw, b.ks, s);
        if (b.nb == 6) return launch_parts<KIND, GROUP, 6>(g, job0, jobs, njobs, blocks, batch, x_raw, b.ks, s);
    }
    if (b.nb == 2) return launch_parts<KIND, GROUP, 2>(g, job0, jobs, njobs, blocks, batch, x_raw, b.ks, s);
    if (b.nb == 4) return launch_parts<KIND, GROUP, 4>(g, job0, jobs, njobs, blocks, batch, x_raw, b.ks, s);
    launch_parts<KIND, GROUP, 8>(g, job0, jobs, njobs, blocks, batch, x_raw, b.ks, s);
}

template <int KIND>
void launch_kind(const CqGeom &g, const CqJob &job0, const CqJob *jobs, int njobs, int blocks, int batch, bool x_raw,
                 hipStream_t s) {
    switch (g.group) {
    case 8: return launch_group<KIND, 8>(g, job0, jobs, njobs, blocks, batch, x_raw, s);
    case 16: return launch_group<KIND, 16>(g, job0, jobs, njobs, blocks, batch, x_raw, s);
    case 32: return launch_group<KIND, 32>(g, job0, jobs, njobs, blocks, batch, x_raw, s);
    default: return launch_group<KIND, 64>(g, job0, jobs, njobs, blocks, batch, x_raw, s);  // 64 and above
    }
}

}  // namespace

}  // namespace nd
