// gfx950 kernels for the int8 KV cache: quantize/store and decode attention.
//
// Store (engine.cpp:1005-1021): per (token, kv head) row, max = absmax,
// scale = max > 0 ? max/127 : 1, inv = max > 0 ? 127/max : 0,
// q = clamp(rint(x * inv), +-127) - multiply by the reciprocal, IEEE
// division for scale and inv, so codes and scales are bit-identical.
//
// Attention (engine.cpp:898-967, 56-74, 137-147, 816-897): for each query
// head h of kv head kh = h / G,
//   s = dot(q_h, float(k_i8)) * k_scale * (1/sqrt(HD))   (sequential over d)
//   p = softmax(s);  out[d] = sum_s (p_s * v_scale_s) * float(v_i8[s][d]).
// In the vector kernel the dot runs over d in the reference's order but with
// fused multiply-adds (one rounding per term instead of two), and the value sums
// likewise; the matrix kernel forms both from exact integer dots. The
// softmax and the value sum are computed split-context (flash decoding):
// each block owns a range of cache slots for one (sequence, kv head) and
// keeps a running max m, a running sum l and unnormalized outputs o; a merge
// pass rescales by exp(m_i - M). That reorders fp32 sums, so results agree
// with the reference to fp32 rounding, not bit for bit.
//
// Device layout (head-major so one (sequence, kv head) context is one
// contiguous run): codes [layer][seq][kvh][capacity][HD] int8, scales
// [layer][seq][kvh][capacity] fp32.
#include "attn.h"
#include "sdot_prepare.h"
#include "wave.h"

#include <cmath>

namespace nd {

namespace {

// One K row and one V row of HD values into the cache, by one wave.
__device__ __forceinline__ void store_kv_row(const float *k, const float *v, int HD, int lane, int8_t *k8, int8_t *v8,
                                             float *ks, float *vs) {
    float mk = 0.0f, mv = 0.0f;
    for (int d = lane; d < HD; d += 64) {
        mk = fmaxf(mk, fabsf(k[d]));
        mv = fmaxf(mv, fabsf(v[d]));
    }
    mk = wave_max(mk, lane);
    mv = wave_max(mv, lane);
    const float sk = mk > 0 ? mk / 127.0f : 1.0f, sv = mv > 0 ? mv / 127.0f : 1.0f;
    const float ik = mk > 0 ? 127.0f / mk : 0.0f, iv = mv > 0 ? 127.0f / mv : 0.0f;
    if (lane == 0) {
        *ks = sk;
        *vs = sv;
    }
    for (int d = lane; d < HD; d += 64) {
        float qk = rintf(k[d] * ik), qv = rintf(v[d] * iv);
        qk = fmaxf(-127.0f, fminf(127.0f, qk));
        qv = fmaxf(-127.0f, fminf(127.0f, qv));
        k8[d] = static_cast<int8_t>(qk);
        v8[d] = static_cast<int8_t>(qv);
    }
}

// One wave per (sequence, token, kv head) row; K and V rows together.
__global__ __launch_bounds__(256) void kv_store_kernel(KvStoreArgs a) {
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    const int rows = a.seqs * a.count * a.kvheads;
    if (wave >= rows) return;
    const int kh = wave % a.kvheads;
    const int i = (wave / a.kvheads) % a.count;
    const int seq = wave / (a.kvheads * a.count);
    const int slot = a.first_slot[seq] + i;
    if (slot < 0 || slot >= a.capacity) return;  // wave-uniform; device-side slot tables are not host-checked
    const size_t src = static_cast<size_t>(wave) * a.head_dim;
    const size_t dst_row = (static_cast<size_t>(seq) * a.kvheads + kh) * a.capacity + slot;
    const int HD = a.head_dim;
    store_kv_row(a.k + src, a.v + src, HD, lane, a.k8 + dst_row * HD, a.v8 + dst_row * HD, a.ks + dst_row,
                 a.vs + dst_row);
}

__device__ __forceinline__ float i8f(uint32_t w, int c) {
    return static_cast<float>(static_cast<int8_t>((w >> (8 * c)) & 0xffu));
}

// With a new token (no slot list, so list position = slot), wave 0 of the
// block whose split holds slot new_slot[seq] (the last split for a slot past
// every range; no block for one outside the cache) first stores the token's K
// and V rows there as kv_store_kernel does; the block barrier (a
// workgroup-scope release and acquire) orders those stores before the block's
// loads of that slot, and no other block reads it. When the slot lies past the
// waves' first sub-tiles, those loads are issued before the store.
template <int HD>
__device__ __forceinline__ void store_new(const AttnArgs &a, int ns, int seq, int kh, size_t row0) {
    if (threadIdx.x < 64) {
        const size_t src = (static_cast<size_t>(seq) * a.kvheads + kh) * HD;
        const size_t dst = row0 + ns;
        store_kv_row(a.new_k + src, a.new_v + src, HD, threadIdx.x, a.k8 + dst * HD, a.v8 + dst * HD, a.ks + dst,
                     a.vs + dst);
    }
    __syncthreads();
}

// The block's result from its four waves' maxima, sums and outputs in LDS (NR
// partial outputs per wave), each wave rescaled to the common maximum: the
// output row (one split; also left prepared as the next projection's input),
// or the split's record.
template <int HD, int G, int NR>
__device__ __forceinline__ void combine_waves(const AttnArgs &a, const float (&lm)[4][G], const float (&ll)[4][G],
                                              const float (&lred)[4][NR][G][HD], int seq, int kh, int sp) {
    const int t = threadIdx.x, lane = t & 63;
    const int H = a.kvheads * G;
    for (int i = t; i < G * HD; i += 256) {
        const int g = i / HD, d = i % HD;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) M = fmaxf(M, lm[w][g]);
        float o = 0.0f, lt = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            if (lm[w][g] == -INFINITY) continue;  // a wave with nothing attended
            const float f = expf(lm[w][g] - M);
            float ow = 0.0f;
            for (int r = 0; r < NR; ++r) ow += lred[w][r][g][d];
            o += f * ow;
            lt += f * ll[w][g];
        }
        const size_t head = static_cast<size_t>(seq) * H + kh * G + g;
        if (a.splits == 1) {
            const float val = lt > 0 ? o * (1.0f / lt) : 0.0f;
            a.out[head * HD + d] = val;
            if (a.prep.q) {
                // whole waves (G * HD is a multiple of 64) over consecutive positions of the sequence's
                // output row: groups of 32 lanes are groups of the next projection's input
                const PrepOut &po = a.prep;
                const int p = (kh * G + g) * HD + d;
                prepare_lane<32>(val, lane, p, po.padded, po.dev, po.scale, po.kind,
                                 po.q + static_cast<size_t>(seq) * po.dev, po.xs + static_cast<size_t>(seq) * po.groups + p / 32,
                                 po.xst + static_cast<size_t>(p / 32) * po.batch + seq);
            }
        } else {
            float *rec = a.part + (head * a.splits + sp) * (HD + 2);
            rec[2 + d] = o;
            if (d == 0) {
                rec[0] = M;
                rec[1] = lt;
            }
        }
    }
}

// Block (split, kv head, sequence): 4 waves, each an independent
// online-softmax worker over 64-slot sub-tiles w, w + 4, w + 8, ... of the
// block's slot range, with the next sub-tile's loads in flight while the
// current one is computed. No block barrier inside the loop; the 4 waves'
// (m, l, o) are combined once at the end.
//   Score phase: lane = slot; the K row is HD/16 16-byte loads; q comes from
//   scalar loads (uniform); dot by fma over d.
//   Value phase: a slot row is HD/4 words, VW words per lane, LPR = HD/4/VW
//   lanes per row, 64/LPR slot lanes, LPR slots per lane per sub-tile.
// All cache reads are buffer loads over this context's rows: a slot that is
// not attended (past the range, or outside [0, capacity) in the caller's
// list) gets an offset past the buffer and reads zero without a memory
// request, so loads need no branches.
template <int HD, bool SLOTS>
__global__ __launch_bounds__(256) void attn_kernel(AttnArgs a) {
    constexpr int G = 1, VW = 4;   // one query head per kv head; 16-byte value loads
    constexpr int DW = HD / 4;
    constexpr int LPR = DW / VW;   // lanes per value row
    constexpr int NLW = 64 / LPR;  // slot lanes per wave
    constexpr int SPL = LPR;       // slots per lane per sub-tile
    constexpr int KC = HD / 16;    // 16-byte chunks per K row
    constexpr uint32_t kOut = 0x80000000u;  // past every buffer (capacity * HD < 2^31)
    static_assert(DW % VW == 0 && 64 % LPR == 0, "value-phase lane mapping");
    __shared__ float lw[4][G][64];
    __shared__ float lred[4][NLW][G][HD];
    __shared__ float lm[4][G], ll[4][G];

    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int sp = blockIdx.x, kh = blockIdx.y, seq = blockIdx.z;
    const int H = a.kvheads * G;
    int len = a.lengths ? a.lengths[seq] : a.length;
    len = len < a.length ? len : a.length;
    const int begin = sp * a.slots_per_split;
    const int end = min(begin + a.slots_per_split, len);
    const uint32_t cap = static_cast<uint32_t>(a.capacity);

    const ND_CONST float *qh = (const ND_CONST float *)(a.q + (static_cast<size_t>(seq) * H + kh * G) * HD);
    const size_t row0 = (static_cast<size_t>(a.shared_cache ? 0 : seq) * a.kvheads + kh) * cap;
    const auto rk = buffer_rsrc(a.k8 + row0 * HD, cap * HD);
    const auto rv = buffer_rsrc(a.v8 + row0 * HD, cap * HD);
    const auto rks = buffer_rsrc(a.ks + row0, cap * 4u);
    const auto rvs = buffer_rsrc(a.vs + row0, cap * 4u);
    const auto rsl = buffer_rsrc(a.slots + static_cast<size_t>(seq) * a.slots_stride, static_cast<uint32_t>(a.length) * 4u);
    const int vj = lane % LPR, vr = lane / LPR;  // value phase: word group, slot lane

    // slot of list position s, or -1 when not attended
    auto slot_of = [&](int s) -> int {
        int raw = s;
        if constexpr (SLOTS) raw = static_cast<int>(__builtin_amdgcn_raw_buffer_load_b32(rsl, s * 4u, 0, 0));
        return (s < end && static_cast<uint32_t>(raw) < cap) ? raw : -1;
    };

    struct Tile {
        u32x4 k[KC];
        uint32_t v[SPL][VW];
        float ks, vs;
        bool valid;
    };
    auto load = [&](Tile &T, int st) {
        const int slot = slot_of(st + lane);
        T.valid = slot >= 0;
        const uint32_t kb = slot >= 0 ? static_cast<uint32_t>(slot) * HD : kOut;
        const uint32_t sb = slot >= 0 ? static_cast<uint32_t>(slot) * 4u : kOut;
#pragma unroll
        for (int c = 0; c < KC; ++c) T.k[c] = __builtin_amdgcn_raw_buffer_load_b128(rk, kb, c * 16, 0);
        T.ks = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rks, sb, 0, 0));
        T.vs = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rvs, sb, 0, 0));
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            const int sv = slot_of(st + vr + i * NLW);
            const uint32_t vb = sv >= 0 ? static_cast<uint32_t>(sv) * HD + vj * VW * 4u : kOut;
            if constexpr (VW == 4) {
                const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(rv, vb, 0, 0);
                T.v[i][0] = w.x;
                T.v[i][1] = w.y;
                T.v[i][2] = w.z;
                T.v[i][3] = w.w;
            } else {
#pragma unroll
                for (int u = 0; u < VW; ++u) T.v[i][u] = __builtin_amdgcn_raw_buffer_load_b32(rv, vb, u * 4, 0);
            }
        }
    };

    float m[G], l[G], acc[G][4 * VW];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        m[g] = -INFINITY;
        l[g] = 0.0f;
#pragma unroll
        for (int c = 0; c < 4 * VW; ++c) acc[g][c] = 0.0f;
    }

    auto compute = [&](const Tile &T) {
        float alpha[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float dot = 0.0f;
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                const uint32_t w4[4] = {T.k[c].x, T.k[c].y, T.k[c].z, T.k[c].w};
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int b = 0; b < 4; ++b) dot = __builtin_fmaf(qh[g * HD + c * 16 + j * 4 + b], i8f(w4[j], b), dot);
            }
            float x = dot * T.ks;
            x *= a.scale;
            x = T.valid ? x : -INFINITY;
            const float mn = fmaxf(m[g], wave_max(x, lane));
            alpha[g] = mn == -INFINITY ? 1.0f : expf(m[g] - mn);
            m[g] = mn;
            const float e = T.valid ? expf(x - mn) : 0.0f;
            l[g] = l[g] * alpha[g] + e;
            lw[wave][g][lane] = e * T.vs;
        }
        // LDS operations of one wave complete in order; the fences only stop
        // the compiler from moving the reads above the writes (and the next
        // sub-tile's writes above these reads).
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int c = 0; c < 4 * VW; ++c) acc[g][c] *= alpha[g];
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const float w = lw[wave][g][vr + i * NLW];
#pragma unroll
                for (int u = 0; u < VW; ++u)
#pragma unroll
                    for (int b = 0; b < 4; ++b) acc[g][u * 4 + b] = __builtin_fmaf(w, i8f(T.v[i][u], b), acc[g][u * 4 + b]);
            }
        }
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
    };

    const int ns = a.new_k ? a.new_slot[seq] : -1;
    const bool store_here =
        a.new_k && ns >= 0 && static_cast<uint32_t>(ns) < cap && sp == min(ns / a.slots_per_split, a.splits - 1);
    const bool store_early = store_here && ns < begin + 256;  // the slot may be in a first sub-tile

    // The next sub-tile is loaded before this one is computed; loads past the
    // end read zero.
    Tile cur, nxt;
    int st = begin + wave * 64;
    if (store_early) store_new<HD>(a, ns, seq, kh, row0);
    load(cur, st);
    if (store_here && !store_early) store_new<HD>(a, ns, seq, kh, row0);
    for (; st < end; st += 256) {
        load(nxt, st + 256);
        asm volatile("" ::: "memory");  // keep the prefetch ahead of the compute
        compute(cur);
        cur = nxt;
    }
    // wave partials -> LDS; combine the 4 waves with their own maxima
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const float ws = wave_sum(l[g], lane);
        if (lane == 0) {
            lm[wave][g] = m[g];
            ll[wave][g] = ws;
        }
#pragma unroll
        for (int c = 0; c < 4 * VW; ++c) lred[wave][vr][g][vj * 4 * VW + c] = acc[g][c];
    }
    __syncthreads();
    combine_waves<HD, G, NLW>(a, lm, ll, lred, seq, kh, sp);
}

// ---- several query heads per kv head: matrix cores on the int8 codes --------
//
// The vector kernel above does every (slot, head, d) term on the VALU, for G
// heads G times (measured at 16 sequences x 8 kv heads x 4 heads x 4096 ragged
// slots of 128: 64 us, 1.4 TB/s of cache). Here both products run on
// v_mfma_i32_16x16x64_i8 (32 deep for rows of 32) straight from the int8
// codes, so the cache stream bounds it: 26.4 us there with the merge pass, 29.6 us
// (4.7 TB/s) at 4096 slots for every sequence.
//
// Both operands are split without loss: two groups of four signed 8-bit digits
// hold 60 bits below the head's largest magnitude. What is left of a q below
// 2^-36 of the largest is multiplied in fp32; weights below 2^-36 get two more
// groups, and again until nothing is left. (28 bits of q and 27 of a weight
// lost the small ones: an outlier in q over zero K codes gave errors of 3e-5 at
// 1e4 times the rest, 4e-3 at 1e6.) The digit dots are exact integers, and
// joining them takes a few roundings relative to the sum of the terms'
// magnitudes, where a chain of fp32 products and sums takes one per term.
//
// Scores. q is split once per block; the 16 rows of operand A are 4 heads x 4
// digits of a group. Operand B is 16 slots' K codes. Output register v of lane l
// is digit v of head l / 16 and slot l % 16, joined in the lane.
//
// Values. w = p * v_scale is split relative to the largest w of the head's 64
// slots, its bytes transposed so that operand A's rows are heads x digits and
// its depth the 64 slots; operand B is the V codes, whose rows a
// lane loads HD / 16 consecutive bytes at a time (lane l: d = HD / 16 *
// (l % 16) ..) for 16 slots and transposes with byte permutes (depth byte
// 4 u + t of lane group l / 16 is slot 16 t + 4 (l / 16) + u). Output register v
// of lane l is digit v of head l / 16, output d = HD / 16 * (l % 16) + i.
// Infinite and NaN weights are multiplied and added slot by slot.
template <int HD>
struct MfmaShape {
    static constexpr int kVB = HD / 16;               // V bytes per lane and slot
    static constexpr int kVD = (kVB + 3) / 4;         // dwords of them
    static constexpr int kKH = HD == 128 ? 2 : 1;     // operand registers of 16 (32: 8) bytes per K row and lane
    static constexpr int kKB = HD == 32 ? 8 : 16;     // bytes of each
};

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x2 __attribute__((ext_vector_type(2)));

template <int HD>
__device__ __forceinline__ i32x4 mfma_rows(const i32x4 &a, const i32x4 &b, const i32x4 &c) {
    if constexpr (HD == 32)
        return __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, i32x2{a.x, a.y}),
                                                     __builtin_bit_cast(long, i32x2{b.x, b.y}), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// Two groups of four digits: x below 2^fe is f1 2^(fe - kFirst) + f2 2^(fe - kSecond) + rest, |f1|, |f2| <= 2^30.
constexpr int kFirst = 30, kSecond = 60;

// The four digits (-128 .. 127, base 256, the lowest first) of f in a dword's bytes.
__device__ __forceinline__ uint32_t digit_bytes(float f) {
    // 128 added to every digit, so that no byte borrows from the next, and taken off each byte again
    return (static_cast<uint32_t>(static_cast<int>(f)) + 0x80808080u) ^ 0x80808080u;
}

// Both groups of x, which keeps the rest. Exact: what a group leaves is at most
// half its unit and has x's own last bit, so it fits fp32, and so does f 2^n (f
// has 24 bits at most from its first to its last).
__device__ __forceinline__ void take_digits(float &x, int fe, uint32_t &y1, uint32_t &y2) {
    const float f1 = rintf(ldexpf(x, kFirst - fe));
    x -= ldexpf(f1, fe - kFirst);
    const float f2 = rintf(ldexpf(x, kSecond - fe));
    x -= ldexpf(f2, fe - kSecond);
    y1 = digit_bytes(f1);
    y2 = digit_bytes(f2);
}

// D0 + D1 2^8 + D2 2^16 + D3 2^24 of integer digit sums |D| <= 2^21.
__device__ __forceinline__ float join_digits(const i32x4 &d) {
    const int hi = d.w * 256 + d.z, lo = d.y * 256 + d.x;
    return __builtin_fmaf(static_cast<float>(hi), 65536.0f, static_cast<float>(lo));
}
// The two groups' digit sums, in units of the first group's last digit.
__device__ __forceinline__ float join_groups(const i32x4 &d1, const i32x4 &d2) {
    return __builtin_fmaf(join_digits(d2), 1.0f / (1 << (kSecond - kFirst)), join_digits(d1));
}

// 4 x 4 byte transpose: out[i] = byte i of in[0], in[1], in[2], in[3].
__device__ __forceinline__ void transpose4(const uint32_t (&in)[4], uint32_t (&out)[4]) {
    const uint32_t a = __builtin_amdgcn_perm(in[1], in[0], 0x05010400u);  // bytes 0, 0, 1, 1 of in[0], in[1]
    const uint32_t b = __builtin_amdgcn_perm(in[1], in[0], 0x07030602u);
    const uint32_t c = __builtin_amdgcn_perm(in[3], in[2], 0x05010400u);
    const uint32_t d = __builtin_amdgcn_perm(in[3], in[2], 0x07030602u);
    out[0] = __builtin_amdgcn_perm(c, a, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(d, b, 0x05040100u);
    out[3] = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

// The larger of v and the butterfly partner's (lane ^ H).
template <int H>
__device__ __forceinline__ uint32_t max_with(uint32_t v, int lane) {
    const uint32_t o = __builtin_bit_cast(uint32_t, butterfly_partner<H>(__builtin_bit_cast(float, v), lane));
    return v > o ? v : o;
}

constexpr uint32_t kInfBits = 0x7F800000u;

// Block and waves as attn_kernel; sub-tiles of 64 slots as four groups t of 16.
// Loads of slots not attended read zero (offsets past the buffer).
template <int HD, int G, bool SLOTS>
__global__ __launch_bounds__(256, 2) void attn_mfma_kernel(AttnArgs a) {
    using S = MfmaShape<HD>;
    constexpr int VB = S::kVB, VD = S::kVD, KH = S::kKH, KB = S::kKB;
    constexpr int HQ = (G + 3) / 4;        // quads of heads
    constexpr int GQ = G < 4 ? G : 4;      // heads of a quad
    constexpr uint32_t kOut = 0x80000000u;  // past every buffer (capacity * HD < 2^31)
    // A operand rows, 16 bytes of row m = 4 head + digit per lane group; a head's four rows are 80 words apart (the
    // writes of the four heads fall in different banks)
    __shared__ __attribute__((aligned(16))) uint32_t wd[4][HQ][2][4 * 80];
    __shared__ __attribute__((aligned(16))) float qrest[4][HQ][GQ][HD];  // what two groups leave of q (each wave its own copy)
    __shared__ float lred[4][1][G][HD];
    __shared__ float lm[4][G], ll[4][G];

    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int col = lane & 15, quad = lane >> 4;  // score lane: slot 16 t + col of head 4 hq + quad
    const int sp = blockIdx.x, kh = blockIdx.y, seq = blockIdx.z;
    const int H = a.kvheads * G;
    int len = a.lengths ? a.lengths[seq] : a.length;
    len = len < a.length ? len : a.length;
    const int begin = sp * a.slots_per_split;
    const int end = min(begin + a.slots_per_split, len);
    const uint32_t cap = static_cast<uint32_t>(a.capacity);

    const float *qh = a.q + (static_cast<size_t>(seq) * H + kh * G) * HD;
    const size_t row0 = (static_cast<size_t>(a.shared_cache ? 0 : seq) * a.kvheads + kh) * cap;
    const auto rk = buffer_rsrc(a.k8 + row0 * HD, cap * HD);
    const auto rv = buffer_rsrc(a.v8 + row0 * HD, cap * HD);
    const auto rks = buffer_rsrc(a.ks + row0, cap * 4u);
    const auto rvs = buffer_rsrc(a.vs + row0, cap * 4u);
    const auto rsl = buffer_rsrc(a.slots + static_cast<size_t>(seq) * a.slots_stride, static_cast<uint32_t>(a.length) * 4u);

    // slot of list position s, or -1 when not attended
    auto slot_of = [&](int s) -> int {
        int raw = s;
        if constexpr (SLOTS) raw = static_cast<int>(__builtin_amdgcn_raw_buffer_load_b32(rsl, s * 4u, 0, 0));
        return (s < end && static_cast<uint32_t>(raw) < cap) ? raw : -1;
    };

    struct Tile {
        i32x4 k[4][KH];
        uint32_t v[4][4][VD];  // [u][t]
        float ks[4], vs[4];
        bool valid[4];
    };
    auto load = [&](Tile &T, int st) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int slot = slot_of(st + 16 * i + col);
            T.valid[i] = slot >= 0;
            const uint32_t kb = slot >= 0 ? static_cast<uint32_t>(slot) * HD + quad * (KB * KH) : kOut;
            const uint32_t sb = slot >= 0 ? static_cast<uint32_t>(slot) * 4u : kOut;
#pragma unroll
            for (int h = 0; h < KH; ++h) {
                if constexpr (KB == 16) {
                    T.k[i][h] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, kb, h * 16, 0));
                } else {
                    const auto w = __builtin_bit_cast(i32x2, __builtin_amdgcn_raw_buffer_load_b64(rk, kb, 0, 0));
                    T.k[i][h] = i32x4{w.x, w.y, 0, 0};
                }
            }
            T.ks[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rks, sb, 0, 0));
            T.vs[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rvs, sb, 0, 0));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int slot = slot_of(st + 16 * i + 4 * quad + u);
                const uint32_t vb = slot >= 0 ? static_cast<uint32_t>(slot) * HD + col * VB : kOut;
                if constexpr (VB == 8) {
                    const auto w = __builtin_bit_cast(i32x2, __builtin_amdgcn_raw_buffer_load_b64(rv, vb, 0, 0));
                    T.v[u][i][0] = w.x;
                    T.v[u][i][VD - 1] = w.y;
                } else if constexpr (VB == 4) {
                    T.v[u][i][0] = __builtin_amdgcn_raw_buffer_load_b32(rv, vb, 0, 0);
                } else {
                    T.v[u][i][0] = static_cast<uint16_t>(__builtin_amdgcn_raw_buffer_load_b16(rv, vb, 0, 0));
                }
            }
    };

    float m[HQ], l[HQ], acc[HQ][VB];
#pragma unroll
    for (int hq = 0; hq < HQ; ++hq) {
        m[hq] = -INFINITY;
        l[hq] = 0.0f;
#pragma unroll
        for (int i = 0; i < VB; ++i) acc[hq][i] = 0.0f;
    }

    const int ns = a.new_k ? a.new_slot[seq] : -1;
    const bool store_here =
        a.new_k && ns >= 0 && static_cast<uint32_t>(ns) < cap && sp == min(ns / a.slots_per_split, a.splits - 1);
    const bool store_early = store_here && ns < begin + 256;  // the slot may be in a first sub-tile
    // q ahead of the tile: its split then runs while the tile is on its way. Lane (head qg, four-value part qj, chunk
    // quad) splits its four values of each chunk.
    const int qg = col >> 2, qj = col & 3;
    const bool qlive = qg < GQ && 4 * qj < KB;
    const int qd = quad * (KB * KH) + 4 * qj;
    float qx[HQ][KH][4];
#pragma unroll
    for (int hq = 0; hq < HQ; ++hq)
#pragma unroll
        for (int h = 0; h < KH; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) qx[hq][h][e] = qlive ? qh[(hq * 4 + qg) * HD + qd + h * KB + e] : 0.0f;
    asm volatile("" ::: "memory");
    Tile cur, nxt;
    int st = begin + wave * 64;
    if (store_early) store_new<HD>(a, ns, seq, kh, row0);
    load(cur, st);
    if (store_here && !store_early) store_new<HD>(a, ns, seq, kh, row0);

    // LDS operations of one wave complete in order; the fences only stop the compiler from moving reads of wd above
    // the writes before them (and later writes above the reads)
    auto lds_fence = [] {
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
    };
    // The lane's operand A of group g from wd: row col = 4 head + digit, lane group quad.
    auto digits = [&](int hq, int g) {
        return *reinterpret_cast<const i32x4 *>(wd[wave][hq][g] + (col >> 2) * 80 + (col & 3) * 16 + quad * 4);
    };

    // q as operand A
    i32x4 q8[HQ][2][KH];
    int qe[HQ];      // of score lane's head: exponent of the first group's last digit
    bool qleft[HQ];  // wave-uniform: qrest is not all zero
    float qscale[HQ];
#pragma unroll
    for (int hq = 0; hq < HQ; ++hq) {
        float (&x)[KH][4] = qx[hq];
        uint32_t top = 0;
#pragma unroll
        for (int h = 0; h < KH; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t bits = __builtin_bit_cast(uint32_t, x[h][e]) & 0x7FFFFFFFu;
                top = top > bits ? top : bits;
            }
        // over the head's sixteen lanes
        top = max_with<1>(top, lane);
        top = max_with<2>(top, lane);
        top = max_with<16>(top, lane);
        top = max_with<32>(top, lane);
        // an infinity or NaN in q makes the head's scores NaN, as its products would
        const bool finite = top < kInfBits;
        const int fe = finite ? __builtin_amdgcn_frexp_expf(__builtin_bit_cast(float, top)) : 0;  // |q| < 2^fe
        qscale[hq] = __shfl(finite ? a.scale : __builtin_nanf(""), 4 * quad);
        qe[hq] = __shfl(fe, 4 * quad) - kFirst;
        bool left = false;
#pragma unroll
        for (int h = 0; h < KH; ++h) {
            uint32_t y1[4], y2[4], z1[4], z2[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[h][e] = finite ? x[h][e] : 0.0f;
                take_digits(x[h][e], fe, y1[e], y2[e]);
                left |= x[h][e] != 0.0f;
            }
            transpose4(y1, z1);  // z[digit]: the four values' bytes
            transpose4(y2, z2);
            const int at = qg * 80 + quad * 4 + qj;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                wd[wave][hq][0][at + i * 16] = z1[i];
                wd[wave][hq][1][at + i * 16] = z2[i];
            }
            lds_fence();
            q8[hq][0][h] = digits(hq, 0);
            q8[hq][1][h] = digits(hq, 1);
            lds_fence();
        }
        qleft[hq] = __any(left);
        if (qleft[hq] && qlive) {
#pragma unroll
            for (int h = 0; h < KH; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) qrest[wave][hq][qg][qd + h * KB + e] = x[h][e];
        }
    }
    lds_fence();

    // Dots of q's two groups with one slot of the tile, in units of the first group's last digit.
    auto score = [&](int hq, const i32x4 (&k)[KH]) {
        i32x4 d1 = {0, 0, 0, 0}, d2 = {0, 0, 0, 0};
#pragma unroll
        for (int h = 0; h < KH; ++h) {
            d1 = mfma_rows<HD>(q8[hq][0][h], k[h], d1);
            d2 = mfma_rows<HD>(q8[hq][1][h], k[h], d2);
        }
        return join_groups(d1, d2);
    };
    // The dot of qrest with list position s's K row (read again).
    auto rest_score = [&](int hq, int s) {
        const int slot = slot_of(s);
        const uint32_t kb = slot >= 0 ? static_cast<uint32_t>(slot) * HD : kOut;
        const float *r = qrest[wave][hq][quad < GQ ? quad : 0];
        float x = 0.0f;
#pragma unroll 1
        for (int d = 0; d < HD; d += 4) {
            const uint32_t w = __builtin_amdgcn_raw_buffer_load_b32(rk, kb + d, 0, 0);
#pragma unroll
            for (int c = 0; c < 4; ++c) x = __builtin_fmaf(r[d + c], i8f(w, c), x);
        }
        return x;
    };

    auto compute = [&](const Tile &T, int st) {
        // V codes as operand B: depth byte 4 u + t
        i32x4 vt[VB];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int w = 0; w < VD; ++w) {
                const uint32_t in[4] = {T.v[u][0][w], T.v[u][1][w], T.v[u][2][w], T.v[u][3][w]};
                uint32_t out[4];
                transpose4(in, out);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (4 * w + i < VB) vt[4 * w + i][u] = static_cast<int>(out[i]);
            }
#pragma unroll
        for (int hq = 0; hq < HQ; ++hq) {
            float x[4];
            float top = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = ldexpf(score(hq, T.k[i]), qe[hq]);
            if (qleft[hq]) {
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] += rest_score(hq, st + 16 * i + col);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] *= T.ks[i];
                x[i] *= qscale[hq];
                x[i] = T.valid[i] ? x[i] : -INFINITY;
                top = fmaxf(top, x[i]);
            }
            const float mn = fmaxf(m[hq], group_max<16>(top, lane));
            const float alpha = mn == -INFINITY ? 1.0f : expf(m[hq] - mn);
            m[hq] = mn;
            float w[4];
            float ls = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float e = T.valid[i] ? expf(x[i] - mn) : 0.0f;
                ls += e;
                w[i] = e * T.vs[i];
            }
            l[hq] = l[hq] * alpha + ls;
#pragma unroll
            for (int i = 0; i < VB; ++i) acc[hq][i] *= alpha;
            // the lane's largest magnitude, as bits
            auto top_bits = [&] {
                uint32_t b = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t bits = __builtin_bit_cast(uint32_t, w[i]) & 0x7FFFFFFFu;
                    b = b > bits ? b : bits;
                }
                return b;
            };
            uint32_t wtop = top_bits();
            if (__any(wtop >= kInfBits)) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
#pragma unroll 1
                    for (int c = 0; c < 16; ++c) {
                        const float ww = __shfl(w[i], quad * 16 + c);
                        if (__builtin_fabsf(ww) < INFINITY) continue;
                        const uint32_t vb = static_cast<uint32_t>(slot_of(st + 16 * i + c)) * HD + col * VB;
#pragma unroll
                        for (int b = 0; b < VB; ++b)
                            acc[hq][b] += ww * i8f(__builtin_amdgcn_raw_buffer_load_b8(rv, vb + b, 0, 0), 0);
                    }
                    w[i] = __builtin_fabsf(w[i]) < INFINITY ? w[i] : 0.0f;
                }
                wtop = top_bits();
            }
            do {
                wtop = max_with<1>(wtop, lane);
                wtop = max_with<2>(wtop, lane);
                wtop = max_with<4>(wtop, lane);
                wtop = max_with<8>(wtop, lane);
                const int fe = __builtin_amdgcn_frexp_expf(__builtin_bit_cast(float, wtop));  // |w| < 2^fe
                uint32_t y1[4], y2[4], z1[4], z2[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) take_digits(w[i], fe, y1[i], y2[i]);
                transpose4(y1, z1);  // z[digit]: bytes t = 0 .. 3
                transpose4(y2, z2);
                const int at = quad * 80 + col;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    wd[wave][hq][0][at + i * 16] = z1[i];
                    wd[wave][hq][1][at + i * 16] = z2[i];
                }
                lds_fence();
                const i32x4 w1 = digits(hq, 0), w2 = digits(hq, 1);
                lds_fence();
                wtop = top_bits();
#pragma unroll
                for (int i = 0; i < VB; ++i) {
                    const i32x4 d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, vt[i], i32x4{0, 0, 0, 0}, 0, 0, 0);
                    const i32x4 d2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(w2, vt[i], i32x4{0, 0, 0, 0}, 0, 0, 0);
                    acc[hq][i] += ldexpf(join_groups(d1, d2), fe - kFirst);
                }
            } while (__any(wtop != 0));
        }
    };

    for (; st < end; st += 256) {
        load(nxt, st + 256);
        asm volatile("" ::: "memory");  // keep the prefetch ahead of the compute
        compute(cur, st);
        cur = nxt;
    }
#pragma unroll
    for (int hq = 0; hq < HQ; ++hq) {
        float ws = l[hq];
        ws += butterfly_partner<1>(ws, lane);
        ws += butterfly_partner<2>(ws, lane);
        ws += butterfly_partner<4>(ws, lane);
        ws += butterfly_partner<8>(ws, lane);
        if (quad < GQ) {
            if (col == 0) {
                lm[wave][hq * 4 + quad] = m[hq];
                ll[wave][hq * 4 + quad] = ws;
            }
#pragma unroll
            for (int i = 0; i < VB; ++i) lred[wave][0][hq * 4 + quad][col * VB + i] = acc[hq][i];
        }
    }
    __syncthreads();
    combine_waves<HD, G, 1>(a, lm, ll, lred, seq, kh, sp);
}

// One block per query head: out = sum_i exp(m_i - M) o_i / sum_i exp(m_i - M) l_i, in split order.
// The records are read kMergeBatch splits at a time, every load of a batch in
// flight together (buffer loads with the whole offset in the range-checked
// lane offset: splits past the count read zero and are skipped), so a merge
// costs one memory round trip per batch, not per split.
constexpr int kMergeBatch = 16;
__global__ __launch_bounds__(128) void attn_merge_kernel(const float *__restrict__ part, float *__restrict__ out,
                                                         int heads_total, int splits, int hd) {
    const int head = blockIdx.x;
    const uint32_t stride = static_cast<uint32_t>(hd + 2) * 4u;  // bytes per split record
    const auto rr = buffer_rsrc(part + static_cast<size_t>(head) * splits * (hd + 2), static_cast<uint32_t>(splits) * stride);
    auto load = [&](int i, int field) {  // field 0: m, 1: l, 2 + d: o[d]
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                             rr, static_cast<uint32_t>(i) * stride + static_cast<uint32_t>(field) * 4u, 0, 0));
    };
    float M = -INFINITY;
    for (int i0 = 0; i0 < splits; i0 += kMergeBatch) {
        float m[kMergeBatch];
#pragma unroll
        for (int k = 0; k < kMergeBatch; ++k) m[k] = load(i0 + k, 0);
#pragma unroll
        for (int k = 0; k < kMergeBatch; ++k)
            if (i0 + k < splits) M = fmaxf(M, m[k]);
    }
    for (int d = threadIdx.x; d < hd; d += blockDim.x) {
        float L = 0.0f, O = 0.0f;
        for (int i0 = 0; i0 < splits; i0 += kMergeBatch) {
            float m[kMergeBatch], l[kMergeBatch], o[kMergeBatch];
#pragma unroll
            for (int k = 0; k < kMergeBatch; ++k) {
                m[k] = load(i0 + k, 0);
                l[k] = load(i0 + k, 1);
                o[k] = load(i0 + k, 2 + d);
            }
#pragma unroll
            for (int k = 0; k < kMergeBatch; ++k) {
                if (i0 + k >= splits || m[k] == -INFINITY) continue;  // past the count, or an empty split
                const float f = expf(m[k] - M);
                L += f * l[k];
                O += f * o[k];
            }
        }
        out[static_cast<size_t>(head) * hd + d] = L > 0 ? O * (1.0f / L) : 0.0f;
    }
}

// One query head per kv head leaves three quarters of the matrix kernel's score
// lanes idle: at rows of 64 the vector kernel is ahead (64 sequences x 8 kv heads
// x 2048 slots 24.4 us; the matrix kernel's two heads take 26.2), at rows of 128
// the matrix kernel in large batches (512 pairs x 600 / 2048 slots 19.0 / 44.8
// against 20.7 / 46.1 us), and its dots of 128 are closer to the exact value.
template <int HD, bool SLOTS>
void launch_attn_hd(const AttnArgs &a, int G, dim3 grid, hipStream_t s) {
    switch (G) {
    case 1:
        if constexpr (HD < 128) hipLaunchKernelGGL((attn_kernel<HD, SLOTS>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((attn_mfma_kernel<HD, 1, SLOTS>), grid, dim3(256), 0, s, a);
        break;
    case 2: hipLaunchKernelGGL((attn_mfma_kernel<HD, 2, SLOTS>), grid, dim3(256), 0, s, a); break;
    case 4: hipLaunchKernelGGL((attn_mfma_kernel<HD, 4, SLOTS>), grid, dim3(256), 0, s, a); break;
    case 8: hipLaunchKernelGGL((attn_mfma_kernel<HD, 8, SLOTS>), grid, dim3(256), 0, s, a); break;
    default: ND_CHECK(false, "attention: heads per kv head must be 1, 2, 4 or 8");
    }
    ND_HIP(hipGetLastError());
}

template <int HD>
void launch_attn_slots(const AttnArgs &a, int G, dim3 grid, hipStream_t s) {
    if (a.slots) launch_attn_hd<HD, true>(a, G, grid, s);
    else launch_attn_hd<HD, false>(a, G, grid, s);
}

}  // namespace

bool attn_supported(int head_dim, int group) {
    return (head_dim == 32 || head_dim == 64 || head_dim == 128) && (group == 1 || group == 2 || group == 4 || group == 8);
}

void launch_kv_store(const KvStoreArgs &a, hipStream_t s) {
    const int rows = a.seqs * a.count * a.kvheads;
    if (rows <= 0) return;
    hipLaunchKernelGGL(kv_store_kernel, dim3((rows + 3) / 4), dim3(256), 0, s, a);
    ND_HIP(hipGetLastError());
}

void launch_attention(AttnArgs a, int group, hipStream_t s) {
    ND_CHECK(attn_supported(a.head_dim, group), "attention: unsupported head_dim / group");
    const int H = a.kvheads * group;
    dim3 grid(a.splits, a.kvheads, a.seqs);
    switch (a.head_dim) {
    case 32: launch_attn_slots<32>(a, group, grid, s); break;
    case 64: launch_attn_slots<64>(a, group, grid, s); break;
    default: launch_attn_slots<128>(a, group, grid, s); break;
    }
    if (a.splits > 1) {
        hipLaunchKernelGGL(attn_merge_kernel, dim3(a.seqs * H), dim3(128), 0, s, a.part, a.out, a.seqs * H, a.splits,
                           a.head_dim);
        ND_HIP(hipGetLastError());
    }
}

}  // namespace nd
