// gfx950 int8 ("SDOT") GEMV of 4-bit codes for 2 to 12 activation rows and
// groups of 32, 64 and 128:
//   value[b][row] += (float(dot_g) * (half(norm) * cs)) * x_scale[b][g]
// for g in group order (sdot.cpp:43-44, 142-149), bit-identical to the
// kernels of sdot_kernels.hip.
//
// What bounds those at a few rows is the VALU: 1.6 instructions a code to turn
// codes into int8 centroids, and four instructions per (weight row, batch row,
// group), for whole quads or sixteens of batch rows. Here
// - codes and activations are multiplied as fp16: integers up to 127 are exact
//   there, their products and sums of a group exact in the fp32
//   accumulators, so the matrix cores deliver float(dot) itself and the
//   epilogue is three instructions for the batch rows there are;
// - a byte of codes is looked up as a pair of fp16 centroids, in a 256-entry
//   LDS table with a column per lane (one v_perm and one conflict-free 4-byte
//   read): half a VALU instruction a code;
// - v_mfma_f32_4x4x4_16b_f16 takes 4 batch rows x 4 positions x 64 weight rows:
//   lane l feeds its own weight row's codes (B) and ends up with its sums, and
//   one register pair holds 4 batch rows x 64 positions of activations (A),
//   block abid broadcast to all by cbsz = 4, so activations are loaded once per
//   64 positions straight from memory and converted there.
#include "common.h"
#include "wave.h"

#include <hip/hip_fp16.h>

#include <type_traits>
#include <utility>

namespace nd {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));

constexpr int kSdBlock = 64;                  // positions handled between two rounds of loads
constexpr int kSdPairTable = 256 * 64;        // dwords of the 4-bit pair table
constexpr int kSdAhead = 4;                   // code dwords looked up ahead of their products
constexpr size_t kSdMaxLds = 160 * 1024;

template <int GROUP, int NB>
struct SdShape {
    static constexpr int kQuads = (NB + 3) / 4;
    static constexpr int kDwords = kSdBlock / 8;  // code dwords per block
    static constexpr int kChunks = kDwords / 4;
    static constexpr int kNorms = GROUP < kSdBlock ? kSdBlock / GROUP : 1;  // groups closing in a block
    static constexpr int kScaleRow = kQuads * 4;                            // floats per group in LDS
};

template <int GROUP, int NB>
struct SdState {
    using S = SdShape<GROUP, NB>;
    u32x4 codes[S::kChunks];
    u32x2v q[S::kQuads];
    uint16_t norms[S::kNorms];
};

// The lane's four activations (batch row l % 4, positions 4 (l / 4) .. + 4 of
// the block) as fp16, from the prepared int8 codes of 8 positions, even ones
// first. A byte b ^ 0x80 under 0x64 is the fp16 number 1024 + 128 + value.
__device__ __forceinline__ h4 sd_halves(const u32x2v &q, uint32_t sel) {
    const uint32_t t = __builtin_amdgcn_perm(q.y, q.x, sel) ^ 0x80808080u;
    const h2v bias = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
    const h2v lo = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, t, 0x04010400u)) + bias;
    const h2v hi = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, t, 0x04030402u)) + bias;
    return h4{lo.x, lo.y, hi.x, hi.y};
}

// fp16 centroid pairs of one code dword, positions in order: byte offset
// 256 * (code byte k) + 4 * lane.
__device__ __forceinline__ void sd_pairs(uint32_t (&v)[4], const uint32_t *table, uint32_t dword, uint32_t lane4) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
        v[k] = *reinterpret_cast<const uint32_t *>(
            reinterpret_cast<const char *>(table) +
            __builtin_amdgcn_perm(dword, lane4, 0x0c0c0400u + (static_cast<uint32_t>(k) << 8)));
}

// Entry e (a byte of codes, low nibble first): 16 stores of 4 columns. A
// thread's entries share the low code, and the high one is the step (no
// indexed read of the arguments).
__device__ __forceinline__ void fill_pair_table(uint32_t *table, const SdotGeom &geom) {
    auto half_of = [&](int code) {  // the code's int8 centroid as fp16
        const int c = static_cast<int8_t>((geom.cent[code >> 2] >> (8 * (code & 3))) & 0xFFu);
        return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<_Float16>(static_cast<float>(c))));
    };
    const int low = threadIdx.x >> 4;
    uint32_t lo = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) lo = low == i ? half_of(i) : lo;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const uint32_t v = lo | half_of(k) << 16;
        reinterpret_cast<u32x4 *>(table)[threadIdx.x + k * kRowsPerBlock] = u32x4{v, v, v, v};
    }
}

template <class F, int... I>
__device__ __forceinline__ void sd_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void sd_for(F &&f) {
    sd_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <int GROUP, int NB>
__device__ __forceinline__ void sd_rows(const SdotJob &J, const SdotGeom &geom, const uint32_t *table,
                                        const float *scales, int blk) {
    using S = SdShape<GROUP, NB>;
    constexpr int NN = S::kNorms, NQ = S::kQuads, D = S::kDwords;
    const int r = threadIdx.x % kRowsPerBlock, lane = threadIdx.x & 63;
    const int tile = blk - J.block_begin;
    const int nb = min(NB, J.batch);
    const int dev = geom.windows * kWindow;  // activation bytes per batch row
    const __amdgpu_buffer_rsrc_t codes =
        buffer_rsrc(J.codes + static_cast<size_t>(tile) * geom.chunks * kRowsPerBlock,
                    static_cast<uint32_t>(geom.chunks) * kRowsPerBlock * 16u);
    const __amdgpu_buffer_rsrc_t norms = buffer_rsrc(J.norms + static_cast<size_t>(tile) * geom.groups * kRowsPerBlock,
                                                     static_cast<uint32_t>(geom.groups) * kRowsPerBlock * 2u);
    const __amdgpu_buffer_rsrc_t acts =
        buffer_rsrc(J.q, static_cast<uint32_t>(nb) * dev);
    const uint32_t code_lane = r * 16u, norm_lane = r * 2u, lane4 = lane * 4u;
    const int bpg_shift = GROUP < kSdBlock ? 0 : __builtin_ctz(geom.group / kSdBlock);
    const int i4 = lane >> 2;  // the lane's positions 4 i4 .. of the block
    uint32_t xv[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q)  // rows past the batch repeat its last row; their outputs are not stored
        xv[q] = static_cast<uint32_t>(min(4 * q + (lane & 3), nb - 1)) * dev + (i4 >> 1) * 8;
    // bytes of the lane's positions in the loaded dwords
    const uint32_t sel = (i4 & 1) ? 0x07030602u : 0x05010400u;
    const int groups = geom.groups;
    const int bpg = 1 << bpg_shift;
    const int blocks = GROUP < kSdBlock ? (groups + NN - 1) / NN : groups << bpg_shift;
    auto load_chunk = [&](int block, int c) {
        return __builtin_amdgcn_raw_buffer_load_b128(
            codes, code_lane, __builtin_amdgcn_readfirstlane((block * S::kChunks + c) * kRowsPerBlock * 16), kStreamLoad);
    };
    auto load_rest = [&](SdState<GROUP, NB> &s, int block) {
        const int so = __builtin_amdgcn_readfirstlane(block * kSdBlock);
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            s.q[q] = __builtin_bit_cast(u32x2v, __builtin_amdgcn_raw_buffer_load_b64(acts, xv[q], so, 0));
#pragma unroll
        for (int k = 0; k < NN; ++k) {  // a group past the last reads zero and is never added
            const int g = GROUP < kSdBlock ? block * NN + k : block >> bpg_shift;
            s.norms[k] = __builtin_amdgcn_raw_buffer_load_b16(
                norms, norm_lane, __builtin_amdgcn_readfirstlane(g * kRowsPerBlock * 2), 0);
        }
    };
    SdState<GROUP, NB> st[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
#pragma unroll
        for (int c = 0; c < S::kChunks; ++c) st[n].codes[c] = load_chunk(n, c);
        load_rest(st[n], n);
    }
    float value[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) value[b] = 0.0f;
    f4 acc[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t w[D][4];  // centroid pairs of the block's code dwords, kSdAhead of them in flight
    static_assert(kSdAhead == 4 && D == 8, "the dwords read ahead are one chunk");
    const u32x4 c0 = st[0].codes[0];
    sd_pairs(w[0], table, c0.x, lane4);
    sd_pairs(w[1], table, c0.y, lane4);
    sd_pairs(w[2], table, c0.z, lane4);
    sd_pairs(w[3], table, c0.w, lane4);

    // closes group g: xs, its activation scales
    auto close = [&](int g, uint16_t norm, const float (&xs)[NQ * 4]) {
        const float ns = __half2float(__ushort_as_half(norm)) * geom.centroid_scale;  // sdot.cpp:43-44
        if (g < groups)
#pragma unroll
            for (int b = 0; b < NB; ++b) value[b] = value[b] + (acc[b / 4][b & 3] * ns) * xs[b];
#pragma unroll
        for (int q = 0; q < NQ; ++q) acc[q] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    // One block: centroid pairs are read four code dwords ahead (a dword is about
    // 60 clocks of work at 8 rows, an LDS read about 130), spent registers are
    // refilled two blocks ahead.
    auto block_step = [&](auto slot, int n) {
        constexpr int cur = decltype(slot)::value;
        SdState<GROUP, NB> &s = st[cur], &t = st[cur ^ 1];
        const int ahead = n + 2;
        float xs[NN][NQ * 4];
#pragma unroll
        for (int k = 0; k < NN; ++k) {
            const int g = min(GROUP < kSdBlock ? n * NN + k : n >> bpg_shift, groups - 1);
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const float4 v = *reinterpret_cast<const float4 *>(scales + g * S::kScaleRow + 4 * q);
                xs[k][4 * q] = v.x;
                xs[k][4 * q + 1] = v.y;
                xs[k][4 * q + 2] = v.z;
                xs[k][4 * q + 3] = v.w;
            }
        }
        h4 a[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) a[q] = sd_halves(s.q[q], sel);
        sd_for<D>([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            constexpr int dn = d + kSdAhead, e = dn & 3;
            const u32x4 &cn = dn < D ? s.codes[dn / 4 % S::kChunks] : t.codes[0];
            sd_pairs(w[dn % D], table, e == 0 ? cn.x : e == 1 ? cn.y : e == 2 ? cn.z : cn.w, lane4);
            if constexpr (d == 0) s.codes[0] = load_chunk(ahead, 0);       // read during the previous block
            if constexpr (dn == D - 1) s.codes[1] = load_chunk(ahead, 1);
            __builtin_amdgcn_sched_barrier(0);
            sd_for<2>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                constexpr int P = 2 * d + i;  // four positions 4 P .. + 4
                const h4 b = __builtin_bit_cast(h4, u32x2v{w[d][2 * i], w[d][2 * i + 1]});
#pragma unroll
                for (int q = 0; q < NQ; ++q) acc[q] = __builtin_amdgcn_mfma_f32_4x4x4f16(a[q], b, acc[q], 4, P, 0);
                if constexpr (GROUP < kSdBlock && 4 * (P + 1) % GROUP == 0)
                    close(n * NN + 4 * (P + 1) / GROUP - 1, s.norms[4 * (P + 1) / GROUP - 1], xs[4 * (P + 1) / GROUP - 1]);
            });
            // pins the dword's products and sums before the next dword's reads
#pragma unroll
            for (int q = 0; q < NQ; ++q) asm volatile("" : "+v"(acc[q]));
#pragma unroll
            for (int b = 0; b < NB; ++b) asm volatile("" : "+v"(value[b]));
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (GROUP >= kSdBlock) {
            if ((n & (bpg - 1)) == bpg - 1) close(n >> bpg_shift, s.norms[0], xs[0]);
        }
        load_rest(s, ahead);
    };
    int n = 0;
    for (; n + 2 <= blocks; n += 2) {
        block_step(std::integral_constant<int, 0>{}, n);
        block_step(std::integral_constant<int, 1>{}, n + 1);
    }
    if (n < blocks) block_step(std::integral_constant<int, 0>{}, n);
    const int row = tile * kRowsPerBlock + r;
    const size_t ys = J.ystride ? J.ystride : J.rows;
    if (row < J.rows) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
            if (b < nb) ((ND_GLOBAL float *)J.y)[static_cast<size_t>(b) * ys + row] = value[b];
    }
}

template <int GROUP, int NB>
__global__ __launch_bounds__(kRowsPerBlock, 2) void sdot_batch_kernel(SdotJob job0, const SdotJob *__restrict__ jobs,
                                                                        int njobs, SdotGeom geom) {
    using S = SdShape<GROUP, NB>;
    // (a static table: its address folds into the lookups)
    __shared__ __attribute__((aligned(16))) uint32_t table[kSdPairTable];
    extern __shared__ __attribute__((aligned(16))) float scales[];  // [groups][kScaleRow]
    const int blk = blockIdx.x;
    SdotJob J = job0;
    if (njobs > 0) {
        const ND_CONST SdotJob *cj = (const ND_CONST SdotJob *)(jobs);
        const int j = find_job(cj, njobs, blk);
        J.codes = cj[j].codes;
        J.norms = cj[j].norms;
        J.q = cj[j].q;
        J.xs = cj[j].xs;
        J.y = cj[j].y;
        J.rows = cj[j].rows;
        J.block_begin = cj[j].block_begin;
        J.batch = cj[j].batch;
        J.ystride = cj[j].ystride;
    }
    fill_pair_table(table, geom);
    const int nb = min(NB, J.batch);
    for (int i = threadIdx.x; i < geom.groups * S::kScaleRow; i += kRowsPerBlock) {
        const int g = i / S::kScaleRow, b = i % S::kScaleRow;
        scales[i] = b < nb ? J.xs[static_cast<size_t>(b) * geom.groups + g] : 0.0f;
    }
    __syncthreads();
    sd_rows<GROUP, NB>(J, geom, table, scales, blk);
}

template <int GROUP, int NB>
bool sd_launch_shape(const SdotGeom &g, const SdotJob &job0, const SdotJob *jobs, int njobs, int blocks, hipStream_t s) {
    using S = SdShape<GROUP, NB>;
    const size_t lds = static_cast<size_t>(g.groups) * S::kScaleRow * 4;
    if (lds + kSdPairTable * 4 > kSdMaxLds) return false;
    const dim3 grid(blocks), block(kRowsPerBlock);
    hipLaunchKernelGGL((sdot_batch_kernel<GROUP, NB>), grid, block, lds, s, job0, jobs, njobs, g);
    ND_HIP(hipGetLastError());
    return true;
}

template <int GROUP>
bool sd_launch_group(const SdotGeom &g, const SdotJob &job0, const SdotJob *jobs, int njobs, int blocks, int batch,
                     hipStream_t s) {
    auto go = [&](auto nb) {
        return sd_launch_shape<GROUP, decltype(nb)::value>(g, job0, jobs, njobs, blocks, s);
    };
    if (batch <= 2) return go(std::integral_constant<int, 2>{});
    if (batch <= 3) return go(std::integral_constant<int, 3>{});
    if (batch <= 4) return go(std::integral_constant<int, 4>{});
    if (batch <= 5) return go(std::integral_constant<int, 5>{});
    if (batch <= 6) return go(std::integral_constant<int, 6>{});
    if (batch <= 8) return go(std::integral_constant<int, 8>{});
    return go(std::integral_constant<int, 12>{});
}

}  // namespace

bool launch_sdot_batch(const SdotGeom &g, const SdotJob &job0, const SdotJob *jobs, int njobs, int blocks, int batch,
                       hipStream_t s) {
    // a group's products of int8 values sum below 2^24; the activations stay below 2^32 bytes
    if (g.kind != kNib || g.group < 32 || g.group > 128 || batch < 2 || batch > 12 || g.windows > 1 << 19) return false;
    if (g.group == 32) return sd_launch_group<32>(g, job0, jobs, njobs, blocks, batch, s);
    return sd_launch_group<64>(g, job0, jobs, njobs, blocks, batch, s);  // 64 and 128
}

}  // namespace nd
