// ml::Attention forward where there are few queries: 32 of them (or the ones there are) per work-group, the keys cut
// between its wavefronts and, where that still leaves the device idle, between work-groups.
//
// The kernels of attention.hip give a wavefront its own queries and let all of a work-group walk the same keys. With one
// query per sequence (tokens being generated) three of their four wavefronts multiply padding, and one work-group has the
// whole key axis of a head to fetch. Here every wavefront fetches and multiplies its own blocks of 32 keys:
//   - blocks are dealt in turn: wavefront w of part z takes w + NW z, then every (NW * parts)-th: with a causal mask too
//     all have the same number of them, to within one;
//   - a wavefront copies its K and V blocks asynchronously into a ring of its own in LDS, S blocks deep, and waits for its
//     own copies only: the loop has no barrier. K of a block and V of a block are separate slots, refilled as soon as
//     they have been read: between 1.5 and 2 blocks of 32 keys (HD * 128 bytes each) are in flight per wavefront, 96-128 KB per CU;
//   - the products are the ones of attention.hip (S^T = K Q^T with a query per lane, O^T += V^T P^T with P straight from
//     the accumulator), and so is the reference point of the exponentials: the first block with a finite score sets it, and it moves only
//     when a row sum shows growth beyond 2^40, an infinity or a NaN. The raw scores of a block are 16 registers here and
//     stay where they are until that is known;
//   - at the end the wavefronts' (m, l, O) meet in LDS: O = sum_w 2^(m_w - M) O_w, l alike, M the largest m_w. With more
//     than one part the work-group writes that unnormalised O, M and l in fp32 and docc_attention_combine_* does the
//     same sum over the parts.
//
// What bounds it: with one query K and V come through once for 4 flop a byte: the memory. A wavefront's MFMAs
// (32 queries a tile, most of them padding) are a tenth of the time its copies take. One query, 16 x 16 heads of 4096 keys
// of 128: 94 us, 5.7 TB/s; 4 heads of 32768 keys: 17 us (in 64 parts) against 609 us with a work-group per head; 4 heads of
// 2048 queries and keys of 64, where a wavefront waits for one block's chain after another: 15 us against 28.
#include "attention.h"

namespace docc_k {

constexpr int kSplitKeys = 32;   // keys per block
constexpr int kSplitQueries = 32;

template <bool OUT_BF16>
__device__ __forceinline__ void store4(void* O, long off, const f32x4& v) {
    if (OUT_BF16) {
        u16x4_t o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = f32_to_bf16_rne(v[e]);
        *reinterpret_cast<u16x4_t*>(reinterpret_cast<uint16_t*>(O) + off) = o;
    } else {
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(O) + off) = v;
    }
}

// the weight of a part whose reference point is m when M is the largest of them (both -inf: nothing finite anywhere, and
// l = 0 or NaN says so in the result)
__device__ __forceinline__ float part_weight(float m, float M) { return M == -__builtin_huge_valf() ? 1.f : __builtin_amdgcn_exp2f(m - M); }

// parts = gridDim.z; parts > 1: `O` is not touched, PO[(head, query), part][HD] and PM[(head, query), part][2] are written
template <bool OUT_BF16, int HD, int NW, int S, bool CAUSAL>
__device__ __forceinline__ void attention_split(const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
                                                const uint16_t* __restrict__ V, void* __restrict__ O, float* __restrict__ PO,
                                                float* __restrict__ PM, int SQ, int SKV, float c) {
    extern __shared__ __attribute__((aligned(16))) unsigned char docc_attn_split_lds[];
    constexpr int kTileElems = kSplitKeys * HD;      // one K or V block, unpadded, 16-byte granules swizzled
    constexpr int GR = HD / 8;                       // granules per row
    constexpr int RP = 64 / GR;                      // rows per copy instruction of the wavefront
    constexpr int P = kSplitKeys / RP;               // copy instructions per block and tensor
    constexpr int KS = HD / 16, DT = HD / 32;
    constexpr int kRowStride = HD + 4;               // floats of a query's O in the exchange: rows start 4 banks apart
    static_assert(NW * S * 2 * kTileElems * 2 >= NW * kSplitQueries * (kRowStride + 2) * 4, "the exchange reuses the ring");
    static_assert(2 * P * S <= 56, "the copies in flight are counted in six bits");

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qj = lane & 31, g = lane >> 5;
    // work-group -> (head, part, query tile): consecutive ids go round the 8 XCDs, renumbered so that an XCD has whole heads
    const int tiles = gridDim.x, parts = gridDim.z, total = gridDim.x * gridDim.y * gridDim.z;
    int lid = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    if (total % 8 == 0) lid = (lid % 8) * (total / 8) + lid / 8;
    const long bh = lid / (tiles * parts);
    const int rest = lid % (tiles * parts);
    const int tile = rest % tiles, part = rest / tiles;
    const int qt0 = tile * kSplitQueries, q = qt0 + qj;
    const int here = SQ - qt0 < kSplitQueries ? SQ - qt0 : kSplitQueries;   // queries of this tile that exist

    const uint16_t* Qh = Q + bh * (long) SQ * HD;
    const char* Kh = reinterpret_cast<const char*>(K + bh * (long) SKV * HD);
    const char* Vh = reinterpret_cast<const char*>(V + bh * (long) SKV * HD);
    const float ninf = -__builtin_huge_valf();

    bf16x8 bq[KS];   // Q^T as the B operand: d = 16 ks + 8 g .. + 7 of query q (an existing row for lanes without a query)
    {
        const uint16_t* row = Qh + (long) (qj < here ? q : qt0) * HD + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) bq[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8_t*>(row + 16 * ks));
    }

    const int seen = CAUSAL && qt0 + here < SKV ? qt0 + here : SKV;          // keys the tile's last query sees
    const int all_blocks = (seen + kSplitKeys - 1) / kSplitKeys;
    const int step = NW * parts, first = wave + NW * part;
    const int n = first < all_blocks ? (all_blocks - first + step - 1) / step : 0;   // this wavefront's blocks

    uint16_t* const ring = reinterpret_cast<uint16_t*>(docc_attn_split_lds) + wave * (S * 2 * kTileElems);
    auto k_slot = [&](int i) { return ring + (i % S) * (2 * kTileElems); };
    auto v_slot = [&](int i) { return ring + (i % S) * (2 * kTileElems) + kTileElems; };
    // LDS granule s (in copy order: lane-contiguous) holds row s / GR, granule column (s % GR) ^ swizzle(row); rows past
    // the last key copy the last key.
    unsigned koff[P], voff[P];   // byte offsets inside a block of the granules that this lane copies
#pragma unroll
    for (int p = 0; p < P; p++) {
        const int row = lane / GR + RP * p;
        koff[p] = (unsigned) (row * (HD * 2) + ((lane % GR) ^ attn_k_swz<HD>(row)) * 16);
        voff[p] = (unsigned) (row * (HD * 2) + ((lane % GR) ^ attn_v_swz<HD>(row)) * 16);
    }
    auto copy = [&](const char* base, uint16_t* slot, int kb, const unsigned (&off)[P], bool may_be_whole) {
        const long key0 = (long) kb * kSplitKeys;
        if (may_be_whole && key0 + kSplitKeys <= SKV) {
            const char* block = base + key0 * (HD * 2);
#pragma unroll
            for (int p = 0; p < P; p++) __builtin_amdgcn_global_load_lds((attn_global_ptr_t) (block + off[p]), (attn_lds_ptr_t) (slot + p * 512), 16, 0, 0);
        } else {
#pragma unroll
            for (int p = 0; p < P; p++) {
                const long key = key0 + lane / GR + RP * p, last = SKV - 1;
                const char* row = base + (key < last ? key : last) * (HD * 2);
                __builtin_amdgcn_global_load_lds((attn_global_ptr_t) (row + off[p] % (HD * 2)), (attn_lds_ptr_t) (slot + p * 512), 16, 0, 0);
            }
        }
    };
    auto copy_k = [&](int i, bool may_be_whole = true) { copy(Kh, k_slot(i), first + i * step, koff, may_be_whole); };
    auto copy_v = [&](int i, bool may_be_whole = true) { copy(Vh, v_slot(i), first + i * step, voff, may_be_whole); };

    f32x16 ot[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) ot[dt][r] = 0.f;
    const f32x16 zero16 = ot[0];
    float m_run = ninf, l_part = 0.f;

    const int ts = lane & 15, tgrp = lane >> 4;                // lane roles of the transposed V reads, as in attention.hip
    const int tr_row = 4 * (tgrp >> 1) + (ts >> 2), tr_col = 16 * (tgrp & 1) + 4 * (ts & 3);
    typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
    bf16x2_t ones;
    ones[0] = (__bf16) 1.0f;
    ones[1] = (__bf16) 1.0f;

    // S blocks on their way; the ones a short run does not have are the last key once more, so that the number of copies is
    // the same for every wavefront and known here. No branch between Q's loads and the wait for them: the compiler would
    // put one for every copy before it.
#pragma unroll
    for (int i = 0; i < S; i++) {
        copy_k(i, false);
        copy_v(i, false);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ks++) asm volatile("s_waitcnt vmcnt(%1)" : "+v"(bq[ks]) : "n"(2 * P * S));
    for (int i = 0; i < n; i++) {
        const int kb = first + i * step;
        const bool steady = i + S < n;
        // K of block i has landed: newer are its V and the S - 1 blocks behind it
        if (steady) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P + 2 * P * (S - 1)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        f32x16 s;
        {
            const uint16_t* ks_ = k_slot(i);
            u16x8_t kv[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ks++) kv[ks] = *reinterpret_cast<const u16x8_t*>(ks_ + attn_k_off<HD>(qj, 2 * ks + g));
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (steady) copy_k(i + S);
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kv[ks]), bq[ks], ks == 0 ? zero16 : s, 0, 0, 0);
        }
        if ((kb + 1) * (long) kSplitKeys > SKV) {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (kb * (long) kSplitKeys + Mfma<float>::acc_row(lane, r) >= SKV) s[r] = ninf;
        }
        if (CAUSAL && kb * kSplitKeys + kSplitKeys - 1 > qt0) {
            const int lim = q - kb * kSplitKeys - 4 * g;       // key = 32 kb + 8 (r / 4) + 4 g + r % 4 > query
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 8 * (r / 4) + (r % 4) > lim ? ninf : s[r];
        }
        auto scaled_max = [&] {
            float mx = s[0];
#pragma unroll
            for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
            return fmaxf(half_swap(mx, 0), half_swap(mx, 1)) * c;
        };
        bf16x2_t pk[8];
        auto exponentials = [&](float m) {
            const float base = m == ninf ? 0.f : m;            // nothing finite yet: p = 0
            float sum = 0.f;
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                bf16x2_t pp;
                pp[0] = (__bf16) __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c, -base));
                pp[1] = (__bf16) __builtin_amdgcn_exp2f(__builtin_fmaf(s[r + 1], c, -base));
                pk[r / 2] = pp;
                sum = __builtin_amdgcn_fdot2_f32_bf16(pp, ones, sum, false);
            }
            return sum;
        };
        // no finite score of this query yet (O and l are 0 then): this block sets the reference point
        if (__builtin_amdgcn_ballot_w64(m_run == ninf) != 0) {
            const float mx = scaled_max();
            m_run = m_run == ninf ? mx : m_run;
        }
        float psum = exponentials(m_run);
        if (__builtin_amdgcn_ballot_w64(!(psum < 0x1p40f)) != 0) {
            const float m_new = fmaxf(m_run, scaled_max());
            const float alpha = m_new == ninf ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            l_part *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) ot[dt][r] *= alpha;
            psum = exponentials(m_new);
        }
        l_part += psum;

        // V of block i has landed: newer are the S - 1 blocks behind it and K of block i + S
        if (steady) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * P * (S - 1) + P) : "memory");
        uint16_t* const vs_ = v_slot(i);
        if ((kb + 1) * (long) kSplitKeys > SKV) {               // 0 * (copied value) must not be a NaN
            const u16x8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
            for (int e = (int) (SKV - kb * (long) kSplitKeys) * GR + lane; e < kSplitKeys * GR; e += 64) *reinterpret_cast<u16x8_t*>(vs_ + e * 8) = z;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        s16x8_t va[2][DT];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int row = 16 * u + tr_row;
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                const int col = 32 * dt + tr_col;
                const uint16_t* plo = vs_ + attn_v_off<HD>(row, col >> 3) + (col & 7);
                const uint16_t* phi = vs_ + attn_v_off<HD>(row + 8, col >> 3) + (col & 7);
                const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*) plo);
                const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*) phi);
                va[u][dt] = s16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (steady) copy_v(i + S);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            struct Pack { bf16x2_t v[4]; } pack = {{pk[4 * u], pk[4 * u + 1], pk[4 * u + 2], pk[4 * u + 3]}};
            const bf16x8 pb = __builtin_bit_cast(bf16x8, pack);
#pragma unroll
            for (int dt = 0; dt < DT; dt++) ot[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, va[u][dt]), pb, ot[dt], 0, 0, 0);
        }
    }

    // the wavefronts' results meet where the rings were: every copy has landed and every read is done
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();
    float* const xo = reinterpret_cast<float*>(docc_attn_split_lds);                 // [NW][32][kRowStride]
    float* const xm = xo + NW * kSplitQueries * kRowStride;                            // [NW][32][2]
    const float l = half_swap(l_part, 0) + half_swap(l_part, 1);
    if (qj < here) {
        float* row = xo + (wave * kSplitQueries + qj) * kRowStride;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int rq = 0; rq < 4; rq++)
                *reinterpret_cast<f32x4*>(row + 32 * dt + 8 * rq + 4 * g) = f32x4{ot[dt][4 * rq], ot[dt][4 * rq + 1], ot[dt][4 * rq + 2], ot[dt][4 * rq + 3]};
        if (g == 0) {
            xm[(wave * kSplitQueries + qj) * 2] = m_run;
            xm[(wave * kSplitQueries + qj) * 2 + 1] = l;
        }
    }
    __syncthreads();
    for (int e = tid; e < here * (HD / 4); e += 64 * NW) {
        const int row = e / (HD / 4), d = (e % (HD / 4)) * 4;
        float M = ninf, L = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) M = fmaxf(M, xm[(w * kSplitQueries + row) * 2]);
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const float f = part_weight(xm[(w * kSplitQueries + row) * 2], M);
            L += f * xm[(w * kSplitQueries + row) * 2 + 1];
            acc += f * *reinterpret_cast<const f32x4*>(xo + (w * kSplitQueries + row) * kRowStride + d);
        }
        const long at = bh * (long) SQ + qt0 + row;
        if (parts == 1) {
            store4<OUT_BF16>(O, at * HD + d, acc * (1.0f / L));
        } else {
            *reinterpret_cast<f32x4*>(PO + (at * parts + part) * HD + d) = acc;
            if (d == 0) {
                PM[(at * parts + part) * 2] = M;
                PM[(at * parts + part) * 2 + 1] = L;
            }
        }
    }
}

// The parts of a row added up, in two steps: a thread takes four values of a row over every G-th part (G a power of two, at most four
// parts each where the work-group is wide enough), then the G sums of a row meet in LDS. A single thread walking 32 parts took 7 us.
template <bool OUT_BF16>
__device__ __forceinline__ void attention_combine(const float* __restrict__ PO, const float* __restrict__ PM, void* __restrict__ O,
                                                  long rows, int HD, int parts, int G) {
    __shared__ f32x4 xa[256];
    __shared__ float xm[256], xl[256];
    const int tid = threadIdx.x, quads = HD / 4, per_row = quads * G;   // 8, 16 or 32 times a power of two, at most 256
    const long row = (long) blockIdx.x * (256 / per_row) + tid / per_row;
    const int grp = tid % per_row / quads, d = tid % quads * 4;
    const float ninf = -__builtin_huge_valf();
    float M = ninf, L = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (row < rows) {
        const float* pm = PM + row * parts * 2;
        const float* po = PO + row * parts * HD + d;
#pragma unroll 4
        for (int p = grp; p < parts; p += G) M = fmaxf(M, pm[2 * p]);
#pragma unroll 4
        for (int p = grp; p < parts; p += G) {
            const float f = part_weight(pm[2 * p], M);
            L += f * pm[2 * p + 1];
            acc += f * *reinterpret_cast<const f32x4*>(po + (long) p * HD);
        }
    }
    if (G > 1) {
        xm[tid] = M;
        xl[tid] = L;
        xa[tid] = acc;
        __syncthreads();
        if (grp != 0) return;
        for (int k = 1; k < G; k++) M = fmaxf(M, xm[tid + k * quads]);
        const float f0 = part_weight(xm[tid], M);
        L *= f0;
        acc *= f0;
        for (int k = 1; k < G; k++) {
            const float f = part_weight(xm[tid + k * quads], M);
            L += f * xl[tid + k * quads];
            acc += f * xa[tid + k * quads];
        }
    }
    if (row < rows) store4<OUT_BF16>(O, row * HD + d, acc * (1.0f / L));
}

} // namespace docc_k

#define DOCC_ATTENTION_SPLIT(name, out_bf16, hd, nw, stages, causal)                                                                \
    extern "C" __global__ __launch_bounds__(64 * nw) void name(const uint16_t* Q, const uint16_t* K, const uint16_t* V, void* O,     \
                                                               float* PO, float* PM, int SQ, int SKV, float scale_log2e) {           \
        docc_k::attention_split<out_bf16, hd, nw, stages, causal>(Q, K, V, O, PO, PM, SQ, SKV, scale_log2e);                         \
    }
#define DOCC_ATTENTION_SPLIT_D(hd, nw, stages)                                                          \
    DOCC_ATTENTION_SPLIT(docc_attention_split_d##hd##_f32out, false, hd, nw, stages, false)              \
    DOCC_ATTENTION_SPLIT(docc_attention_split_d##hd##_bf16out, true, hd, nw, stages, false)              \
    DOCC_ATTENTION_SPLIT(docc_attention_split_d##hd##_f32out_causal, false, hd, nw, stages, true)        \
    DOCC_ATTENTION_SPLIT(docc_attention_split_d##hd##_bf16out_causal, true, hd, nw, stages, true)

// LDS: 4 wavefronts x S blocks x HD * 128 bytes (keep in step with the launcher)
DOCC_ATTENTION_SPLIT_D(32, 4, 4)
DOCC_ATTENTION_SPLIT_D(64, 4, 2)
DOCC_ATTENTION_SPLIT_D(128, 4, 2)

extern "C" __global__ __launch_bounds__(256) void docc_attention_combine_f32out(const float* PO, const float* PM, void* O, long rows, int HD, int parts, int G) {
    docc_k::attention_combine<false>(PO, PM, O, rows, HD, parts, G);
}
extern "C" __global__ __launch_bounds__(256) void docc_attention_combine_bf16out(const float* PO, const float* PM, void* O, long rows, int HD, int parts, int G) {
    docc_k::attention_combine<true>(PO, PM, O, rows, HD, parts, G);
}
