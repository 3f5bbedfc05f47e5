// ah_few.hip -- prefill GEMM for a few tokens (sequences decoded together, a drafted run, a short
// prompt): every GGUF family, optionally with the FFN's SwiGLU epilogue.
//
// Reference semantics as ah_gemm.hip: column c of matmat_q8act (kern/matmat.rs:134) is matvec_q8act
// on token c.  At 2 to 32 tokens the weights are still read once per call, as in a GEMV, and what
// bounds the call is latency: the operand pass, the K loop of a tile made for 64 or 128 tokens and
// the split-K reduction were three dependent launches of 4 to 23 us each.  Here one launch does all
// of it.  A workgroup is up to 16 waves: S along K (ah_few_splits) for each of R row tiles of 16
// weight rows, 5 to 8 waves where S is below 8; with the SwiGLU epilogue four row tiles, 4 S waves.
//   * The workgroup quantizes its tokens' activations into LDS itself (the GEMV's quantizer; a
//     QuantAct input is copied), so no operand pass runs before it.
//   * A wave takes its K range a unit (128 or 256 K) at a time, the next unit's weight bytes in flight
//     in registers, and forms each 32-block's exact integer dots with one
//     v_mfma_i32_16x16x32_i8 (codes of 16 tokens x 16 rows; families with a scale per 16 elements
//     use two, with one half of the weight lanes masked each).  Each block's dots fold in f32 with
//     the token's own block scale and the row's scale, as the GEMV folds them, so no exponent band
//     applies and no token needs an exact path.
//   * The S partial sums of a row tile meet in LDS in a fixed order: no partials in memory.
// The int8 fold is 3 to 5 VALU instructions an element and block, which a large tile could not
// afford (ah_gemm.hip's f16 operands fold once a super-block); at one or two token tiles it is a
// few hundred cycles in all.
// Measured on MI355X: the FFN of 8 tokens at 1536 / 8960 (Q4_K gate and up, Q6_K down) 53.9 -> 27.7 us
// in two launches instead of seven; Q5_0 4861 x 901 at 5 tokens 19.4 -> 7.5 us;
// Q6_K 1536 x 8960 at 16 tokens 33.3 -> 16.6 us from codes.
#include "ah_internal.h"
#include "ah_few.h"
#include "ah_swiglu.h"
#include "ah_units.h"

namespace {

typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kOob = 0xFFFFFFF0u;  // past any payload (payloads stay below 4 GiB - 256)

AH_DEV v4i32 dot32(u32x2 a, u32x2 b) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b),
                                                 (v4i32){0, 0, 0, 0}, 0, 0, 0);
}
// bytes u (below 128) minus 2^B, as signed bytes: no byte borrows with its bit 7 set, and adding
// 128 back is that bit flipped
template <int B>
AH_DEV u32x2 sub_top(u32x2 u) {
    constexpr uint32_t one = 0x01010101u << B;
    return (u32x2){((u.x | 0x80808080u) - one) ^ 0x80808080u, ((u.y | 0x80808080u) - one) ^ 0x80808080u};
}

// The workgroup's quantized tokens in LDS.  Codes rows are kpad + 16 bytes apart, so the 16 tokens
// of a fragment read (8 bytes each) fall in different banks; scales are [block][ntp] so that one
// 16-byte read gives a lane its four tokens.
constexpr uint32_t kRowPad = 16;
struct FewAct {
    uint8_t *codes;
    float *fsc;  // [kpad / 32][ntp] S_b * 2^-32
    float *fx;   // Q4_K: [kpad / 32][ntp] fsc * X; Q2_K: [kpad / 16][ntp] fsc * (16-group sum)
    uint32_t stride, ntp;
};

template <int TYPE>
AH_DEV void stage_f32(const FewArgs &a, const FewAct &A, uint32_t tok0, uint32_t ntile) {
    const uint32_t nbp = a.kpad / 32, q = threadIdx.x & 3u;
    const uint32_t quads = ntile * nbp, per = blockDim.x / 4;
    const __amdgpu_buffer_rsrc_t rx = ah_rsrc(a.x, a.n_tok * a.n_in * 4u);
    auto load = [&](uint32_t i) {
        const uint32_t t = i / nbp, b = i - t * nbp, k0 = 32 * b + 8 * q, row = (tok0 + t) * a.n_in;
        QuadIn in;
        in.take = i < quads && a.n_in > k0 ? (a.n_in - k0 < 8 ? a.n_in - k0 : 8) : 0;
        in.s0 = in.s1 = 0;
#pragma unroll
        for (int j = 8; j < 16; ++j) in.w[j] = 0;
        const u32x4 l0 = ah_ld128(rx, in.take ? 4 * (row + k0) : kOob), l1 = ah_ld128(rx, in.take ? 4 * (row + k0) + 16 : kOob);
        in.w[0] = l0.x; in.w[1] = l0.y; in.w[2] = l0.z; in.w[3] = l0.w;
        in.w[4] = l1.x; in.w[5] = l1.y; in.w[6] = l1.z; in.w[7] = l1.w;
        return in;
    };
    QuadIn next = load(threadIdx.x / 4);
    for (uint32_t base = 0; base < quads; base += per) {
        const uint32_t i = base + threadIdx.x / 4;
        QuadIn in = next;
        if (base + per < quads) next = load(i + per);
        if (a.n_in % 32) {  // the words past a ragged row are the next token's
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) in.w[j] = j < in.take ? in.w[j] : 0u;
        }
        const uint32_t t = i / nbp, b = i - t * nbp;
        const QuadOut o = quad_quant(in, AH_SRC_F32, b, a.status, (unsigned long long)(tok0 + t) * a.n_in);
        if (i >= quads) continue;
        *reinterpret_cast<u32x2 *>(A.codes + t * A.stride + 32 * b + 8 * q) = (u32x2){o.c0, o.c1};
        if (q == 0) A.fsc[b * A.ntp + t] = o.fsc;
        if constexpr (TYPE == AH_GGML_Q4_K) {
            if (q == 2) A.fx[b * A.ntp + t] = o.fsc * (float)o.s32;
        } else if constexpr (TYPE == AH_GGML_Q2_K) {
            if (q & 1u) A.fx[(2 * b + (q >> 1)) * A.ntp + t] = o.fsc * (float)o.s16;
        }
    }
}

// A QuantAct's tokens: a lane takes 16 codes and their block's scale, kBatch of them in flight.  Rows
// off the dword grid are read as the dwords that hold them, 16 bytes and one dword, and shifted: a
// load a byte took 4861 x 901 of Q5_0 at 5 tokens 10.6 us (now 9.2), 1536 x 4865 of Q4_K at 16 tokens
// 34.3 us (now 13.9).
template <int TYPE, bool UNALIGNED>
AH_DEV void stage_codes(const FewArgs &a, const FewAct &A, uint32_t tok0, uint32_t ntile) {
    constexpr uint32_t kBatch = UNALIGNED ? 3 : 4;  // (4 would take the kernel past 80 VGPRs, a wave a SIMD less)
    const uint32_t off = UNALIGNED ? (uint32_t)reinterpret_cast<uintptr_t>(a.x) & 3u : 0u;
    const uint32_t nch = a.kpad / 16, nb32 = (a.n_in + 31) / 32, total = ntile * nch;
    const __amdgpu_buffer_rsrc_t rx = ah_rsrc(static_cast<const uint8_t *>(a.x) - off, a.n_tok * a.pitch + off), rsc = ah_rsrc(a.scales, a.n_tok * nb32 * 8u);
    for (uint32_t base = 0; base < total; base += kBatch * blockDim.x) {
        u32x4 c[kBatch];
        u32x2 s[kBatch];
        uint32_t tt[kBatch], kk[kBatch];
        [[maybe_unused]] uint32_t past[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t i = base + j * blockDim.x + threadIdx.x;
            const uint32_t t = i / nch, k = 16 * (i - t * nch);
            const bool in = i < total && k < a.n_in;
            tt[j] = t;
            kk[j] = k;
            const uint32_t at = (tok0 + t) * a.pitch + k + off;
            c[j] = ah_ld128(rx, in ? (UNALIGNED ? at & ~3u : at) : kOob);
            if constexpr (UNALIGNED) past[j] = ah_ld32(rx, in ? (at & ~3u) + 16 : kOob);
            s[j] = ah_ld64(rsc, in ? 8 * ((tok0 + t) * nb32 + k / 32) : kOob);
        }
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t i = base + j * blockDim.x + threadIdx.x, t = tt[j], k = kk[j];
            const uint32_t take = i < total && k < a.n_in ? (a.n_in - k < 16 ? a.n_in - k : 16) : 0;
            uint32_t w[4] = {c[j].x, c[j].y, c[j].z, c[j].w};
            if constexpr (UNALIGNED) {
                const uint32_t sh = ((tok0 + t) * a.pitch + k + off) & 3u;
                w[0] = ah_alignbyte(w[1], w[0], sh);
                w[1] = ah_alignbyte(w[2], w[1], sh);
                w[2] = ah_alignbyte(w[3], w[2], sh);
                w[3] = ah_alignbyte(past[j], w[3], sh);
            }
#pragma unroll
            for (uint32_t x = 0; x < 4; ++x)  // bytes past n_in are the next token's
                w[x] = take >= 4 * x + 4 ? w[x] : take <= 4 * x ? 0u : w[x] & ((1u << (8 * (take - 4 * x))) - 1u);
            const int64_t S = (int64_t)(((uint64_t)s[j].y << 32) | s[j].x);
            // QuantAct::dequantizes (chart/mod.rs:128-134), as quad_quant checks it
            const uint64_t mag = S < 0 ? 0ull - (uint64_t)S : (uint64_t)S;
            if (__builtin_amdgcn_ballot_w64(mag > (1ull << 56)) != 0ull) {
                bool bad = false;
#pragma unroll
                for (uint32_t e = 0; e < 16; ++e) {
                    int64_t prod;
                    bad |= __builtin_mul_overflow(S, (int64_t)(int8_t)((w[e / 4] >> (8 * (e & 3u))) & 0xffu), &prod);
                }
                if (bad) ah_record(a.status, AH_QUANT_ORDER_BASE + ((((unsigned long long)(tok0 + t) * a.n_in >> 5) + k / 32) << 8) + 7u);
            }
            const float fsc = (float)S * 0x1p-32f;
            int s16 = 0;
            if constexpr (TYPE == AH_GGML_Q4_K || TYPE == AH_GGML_Q2_K) {
#pragma unroll
                for (uint32_t x = 0; x < 4; ++x) s16 = ah_sdot4(0x01010101u, w[x], s16);
            }
            const int s32 = TYPE == AH_GGML_Q4_K ? s16 + (int)quad_xor1((uint32_t)s16) : 0;
            if (i >= total) continue;
            *reinterpret_cast<u32x4 *>(A.codes + t * A.stride + k) = (u32x4){w[0], w[1], w[2], w[3]};
            if ((k & 16u) == 0) {
                A.fsc[k / 32 * A.ntp + t] = fsc;
                if constexpr (TYPE == AH_GGML_Q4_K) A.fx[k / 32 * A.ntp + t] = fsc * (float)s32;
            }
            if constexpr (TYPE == AH_GGML_Q2_K) A.fx[k / 16 * A.ntp + t] = fsc * (float)s16;
        }
    }
}

// A wave streams its 16 rows a unit at a time (256 K of a K-quant, 128 K of the 32-block families):
// the unit's bytes of every row are read with 16-byte loads in which consecutive lanes take
// consecutive chunks of a row (whole cache lines, used once), wait in registers while the unit
// before is computed, and go through the wave's own LDS slot, [16 rows][kPitch], an odd multiple of
// 16 bytes so that the 16 rows of a fragment read fall in different banks.  (Reading the fragments
// straight from memory fetched each line several times: 15.8 against 10.9 us at 1536 x 8960.)
template <int TYPE>
struct Unit {
    static constexpr uint32_t k = ah_blk32(TYPE) ? 128u : 256u;
    static constexpr uint32_t bytes = TYPE == AH_GGML_Q8_0 ? 136u : TYPE == AH_GGML_Q5_0 ? 88u : TYPE == AH_GGML_Q4_K ? 144u
                                    : TYPE == AH_GGML_Q6_K ? 210u : TYPE == AH_GGML_Q2_K ? 84u : 110u;
    // chunks of a row's unit from the 16-aligned address below it (Q4_K rows are 16-aligned)
    static constexpr uint32_t chunks = (bytes + (TYPE == AH_GGML_Q4_K ? 0u : 14u) + 15u) / 16u;
    static constexpr uint32_t pitch = 16u * (chunks | 1u);
    static constexpr uint32_t loads = (16u * chunks + 63u) / 64u;
    static constexpr uint32_t slot = 16u * pitch;
};
uint32_t unit_k_of(uint32_t type) { return ah_blk32((int)type) ? 128u : 256u; }
uint32_t slot_of(uint32_t type) {
    switch (type) {
    case AH_GGML_Q8_0: return Unit<AH_GGML_Q8_0>::slot;
    case AH_GGML_Q5_0: return Unit<AH_GGML_Q5_0>::slot;
    case AH_GGML_Q2_K: return Unit<AH_GGML_Q2_K>::slot;
    case AH_GGML_Q3_K: return Unit<AH_GGML_Q3_K>::slot;
    case AH_GGML_Q4_K: return Unit<AH_GGML_Q4_K>::slot;
    default: return Unit<AH_GGML_Q6_K>::slot;
    }
}
// 8 bytes at a 2-aligned offset of the slot
AH_DEV u32x2 lds8(const uint8_t *s, uint32_t x) {
    const uint32_t *p = reinterpret_cast<const uint32_t *>(s + (x & ~3u));
    return (u32x2){ah_alignbyte(p[1], p[0], x & 3u), ah_alignbyte(p[2], p[1], x & 3u)};
}
AH_DEV uint32_t lds2(const uint8_t *s, uint32_t x) {
    return (*reinterpret_cast<const uint32_t *>(s + (x & ~3u)) >> (8 * (x & 3u))) & 0xffffu;
}

// One wave's sums over its units: acc[j][r] is token 16 j + 4 kg + r of the tile, row n.
template <int TYPE, int NT>
struct FewWave {
    typedef Unit<TYPE> U;
    __amdgpu_buffer_rsrc_t rs;
    uint32_t n_in, n, kg, u1;
    uint32_t rb;                // the lane's own row (n)
    uint32_t src[U::loads];     // row offsets of the lane's chunks (kOob: none)
    uint32_t col[U::loads];     // their chunk indexes
    uint32_t dst[U::loads];     // their slot offsets
    uint32_t tok[NT], grp[NT];  // the lane's operand token and first scale token, inside the tile
    u32x4 w[U::loads];
    float acc[NT][4];

    AH_DEV void plan(uint32_t row0, uint32_t n_out, uint32_t row_bytes, uint32_t lane) {
#pragma unroll
        for (uint32_t i = 0; i < U::loads; ++i) {
            const uint32_t c = lane + 64 * i, r = c / U::chunks;
            col[i] = c - r * U::chunks;
            src[i] = r < 16 && row0 + r < n_out ? (row0 + r) * row_bytes : kOob;
            dst[i] = r < 16 ? r * U::pitch + 16 * col[i] : 0u;
        }
    }
    AH_DEV void load(uint32_t u) {
#pragma unroll
        for (uint32_t i = 0; i < U::loads; ++i)
            w[i] = ah_ld128_nt(rs, src[i] != kOob ? ((src[i] + u * U::bytes) & ~15u) + 16 * col[i] : kOob);
    }
    AH_DEV void stage(uint8_t *slot, uint32_t lane) const {
#pragma unroll
        for (uint32_t i = 0; i < U::loads; ++i)
            if (16 * U::chunks >= 64 * (i + 1) || lane + 64 * i < 16 * U::chunks) *reinterpret_cast<u32x4 *>(slot + dst[i]) = w[i];
    }

    AH_DEV u32x2 codes(const FewAct &A, int j, uint32_t k) const {
        return *reinterpret_cast<const u32x2 *>(A.codes + tok[j] * A.stride + k + 8 * kg);
    }
    AH_DEV f32x4 four(const float *p, const FewAct &A, int j, uint32_t b) const {
        return *reinterpret_cast<const f32x4 *>(p + b * A.ntp + grp[j]);
    }
    // A unit's sums are formed apart and join acc once (a K-quant's with d and dmin): the integer
    // products are exact in f32, so a block costs one rounding, as in the GEMV's units.
    typedef float Sums[NT][4];
    // a 32-block with its own scale: s += S * (d * D), D its dots
    AH_DEV void block(const FewAct &A, Sums &s, uint32_t b, u32x2 q, float d) const {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const v4i32 D = dot32(codes(A, j, 32 * b), q);
            const f32x4 fs = four(A.fsc, A, j, b);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[j][r] = __builtin_fmaf(fs[r], d * (float)D[r], s[j][r]);
        }
    }
    // a sub-block of a super-block: s += S * (sc * D) (below 2^22)
    AH_DEV void block_sc(const FewAct &A, Sums &s, uint32_t b, u32x2 q, int sc) const {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const v4i32 D = dot32(codes(A, j, 32 * b), q);
            const f32x4 fs = four(A.fsc, A, j, b);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[j][r] = __builtin_fmaf(fs[r], (float)__mul24(sc, D[r]), s[j][r]);
        }
    }
    // a 32-block of a super-block with a scale per 16 elements: its two dots weighted as one integer
    AH_DEV void block16(const FewAct &A, Sums &s, uint32_t b, u32x2 q, int sc0, int sc1) const {
        const uint32_t m0 = kg < 2 ? 0xFFFFFFFFu : 0u;
        const u32x2 q0 = {q.x & m0, q.y & m0}, q1 = {q.x & ~m0, q.y & ~m0};
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const u32x2 x = codes(A, j, 32 * b);
            const v4i32 D0 = dot32(x, q0), D1 = dot32(x, q1);
            const f32x4 fs = four(A.fsc, A, j, b);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                s[j][r] = __builtin_fmaf(fs[r], (float)(__mul24(sc0, D0[r]) + __mul24(sc1, D1[r])), s[j][r]);
        }
    }
    // s += m * fx: a min over block (or 16-group) b
    AH_DEV void mins(const FewAct &A, Sums &s, uint32_t b, float m) const {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const f32x4 fx = four(A.fx, A, j, b);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[j][r] = __builtin_fmaf(m, fx[r], s[j][r]);
        }
    }
    AH_DEV void add(const Sums &s, float d) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[j][r] = __builtin_fmaf(d, s[j][r], acc[j][r]);
    }

    // unit u from the slot; lane (n, kg) takes elements 8 kg .. 8 kg + 7 of each 32-block of row n
    AH_DEV void compute(const FewAct &A, const uint8_t *slot, uint32_t u) {
        const uint8_t *p = slot + n * U::pitch;
        const uint32_t x = (rb + u * U::bytes) & 15u;  // the unit's first byte in its chunks
        Sums sd = {}, sm = {};
        if constexpr (TYPE == AH_GGML_Q8_0) {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t b = 4 * u + j;
                // (past the row's blocks lie other rows' bytes: no scale is read from them)
                const float d = 32 * b < n_in ? ah_f16_bits_to_f32(lds2(p, x + 34 * j)) : 0.0f;
                block(A, sd, b, lds8(p, x + 34 * j + 2 + 8 * kg), d);
            }
            add(sd, 1.0f);
        } else if constexpr (TYPE == AH_GGML_Q5_0) {
            // lane group kg holds outputs 8 kg ..: the low (kg < 2) or high nibbles of qs[8 (kg & 1) ..]
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t b = 4 * u + j, sh = kg < 2 ? 0u : 4u;
                const float d = 32 * b < n_in ? ah_f16_bits_to_f32(lds2(p, x + 22 * j)) : 0.0f;
                const uint32_t qh = lds2(p, x + 22 * j + 2 + (kg & 2u)) >> (8 * (kg & 1u));
                u32x2 q = lds8(p, x + 22 * j + 6 + 8 * (kg & 1u));
                q.x = ((q.x >> sh) & 0x0F0F0F0Fu) | ((((qh & 0xFu) * 0x00204081u) & 0x01010101u) << 4);
                q.y = ((q.y >> sh) & 0x0F0F0F0Fu) | (((((qh >> 4) & 0xFu) * 0x00204081u) & 0x01010101u) << 4);
                block(A, sd, b, sub_top<4>(q), d);
            }
            add(sd, 1.0f);
        } else if constexpr (TYPE == AH_GGML_Q4_K) {
            const u32x4 h = *reinterpret_cast<const u32x4 *>(p);
            const float fd = ah_f16_bits_to_f32(h.x & 0xffffu), fdm = ah_f16_bits_to_f32(h.x >> 16);
            const Q4kScales q4 = q4k_scales(h.y, h.z, h.w);
#pragma unroll
            for (uint32_t P = 0; P < 4; ++P) {
                if (256 * u + 64 * P >= n_in) break;  // (uniform: a ragged row's last pairs)
                const u32x2 qs = *reinterpret_cast<const u32x2 *>(p + 16 + 32 * P + 8 * kg);
#pragma unroll
                for (uint32_t j = 0; j < 2; ++j) {
                    const uint32_t b = 8 * u + 2 * P + j, at = (2 * P + j) & 3u;
                    const u32x2 q = {(qs.x >> (4 * j)) & 0x0F0F0F0Fu, (qs.y >> (4 * j)) & 0x0F0F0F0Fu};
                    block_sc(A, sd, b, q, q4k_byte(q4.sc[P >> 1], at));
                    mins(A, sm, b, (float)q4k_byte(q4.m[P >> 1], at));
                }
            }
            add(sd, fd);
            add(sm, -fdm);
        } else if constexpr (TYPE == AH_GGML_Q6_K) {
            const float d = ah_f16_bits_to_f32(lds2(p, x + 208));
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                if (256 * u + 128 * h >= n_in) break;
                const u32x2 ql[2] = {lds8(p, x + 64 * h + 8 * kg), lds8(p, x + 64 * h + 32 + 8 * kg)};
                const u32x2 qh = lds8(p, x + 128 + 32 * h + 8 * kg), sc = lds8(p, x + 192 + 8 * h);
#pragma unroll
                for (uint32_t t = 0; t < 4; ++t) {
                    const u32x2 l = ql[t & 1];
                    u32x2 v;
                    v.x = ((t < 2 ? l.x : l.x >> 4) & 0x0F0F0F0Fu) | (((qh.x >> (2 * t)) & 0x03030303u) << 4);
                    v.y = ((t < 2 ? l.y : l.y >> 4) & 0x0F0F0F0Fu) | (((qh.y >> (2 * t)) & 0x03030303u) << 4);
                    const uint32_t s2 = (t < 2 ? sc.x : sc.y) >> (16 * (t & 1));
                    block16(A, sd, 8 * u + 4 * h + t, sub_top<5>(v), (int)(int8_t)(s2 & 0xffu), (int)(int8_t)((s2 >> 8) & 0xffu));
                }
            }
            add(sd, d);
        } else {
            constexpr bool Q3 = TYPE == AH_GGML_Q3_K;
            const float d = ah_f16_bits_to_f32(lds2(p, x + (Q3 ? 108 : 80))), dm = Q3 ? 0.0f : ah_f16_bits_to_f32(lds2(p, x + 82));
            const u32x2 hm = Q3 ? lds8(p, x + 8 * kg) : (u32x2){0u, 0u};
            const u32x2 s01 = Q3 ? lds8(p, x + 96) : (u32x2){0u, 0u};
            const uint32_t s2w = Q3 ? lds2(p, x + 104) | (lds2(p, x + 106) << 16) : 0u;
#pragma unroll
            for (uint32_t h = 0; h < 2; ++h) {
                if (256 * u + 128 * h >= n_in) break;
                const u32x2 qs = lds8(p, x + (Q3 ? 32 : 16) + 32 * h + 8 * kg);
                // Q3_K: the half's 6-bit scales, groups 0-3 and 4-7 (unit_k23); Q2_K: its (sc, m) bytes
                const u32x2 sw = Q3 ? (u32x2){((s01.x >> (4 * h)) & 0x0F0F0F0Fu) | (((s2w >> (4 * h)) & 0x03030303u) << 4),
                                              ((s01.y >> (4 * h)) & 0x0F0F0F0Fu) | (((s2w >> (4 * h + 2)) & 0x03030303u) << 4)}
                                    : lds8(p, x + 8 * h);
#pragma unroll
                for (uint32_t r = 0; r < 4; ++r) {
                    const uint32_t b = 8 * u + 4 * h + r, s2 = (r < 2 ? sw.x : sw.y) >> (16 * (r & 1));
                    u32x2 v = {(qs.x >> (2 * r)) & 0x03030303u, (qs.y >> (2 * r)) & 0x03030303u};
                    if constexpr (Q3) {
                        v.x |= ((hm.x >> (4 * h + r)) & 0x01010101u) << 2;
                        v.y |= ((hm.y >> (4 * h + r)) & 0x01010101u) << 2;
                        block16(A, sd, b, sub_top<2>(v), (int)(s2 & 0xffu) - 32, (int)((s2 >> 8) & 0xffu) - 32);
                    } else {
                        block16(A, sd, b, v, (int)(s2 & 15u), (int)((s2 >> 8) & 15u));
                        mins(A, sm, 2 * b, (float)((s2 >> 4) & 15u));
                        mins(A, sm, 2 * b + 1, (float)((s2 >> 12) & 15u));
                    }
                }
            }
            add(sd, d);
            if constexpr (!Q3) add(sm, -dm);
        }
    }
};

template <int TYPE, int NT, bool FFN>
__global__ void __launch_bounds__(64 * kFewMaxWaves) gemm_few_kernel(FewArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    // XCD-aware order: the token tiles of a row group run on one XCD and share its L2
    const uint32_t per = gridDim.x >> 3;
    const uint32_t L = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (L >= a.n_wg) return;
    uint32_t pi = 0;
#pragma unroll
    for (uint32_t i = 1; i < kFewMaxParts; ++i)
        if (!FFN && i < a.n_parts && L >= a.p[i].wg_begin) pi = i;
    const uint32_t Lp = L - (FFN ? 0u : a.p[pi].wg_begin);
    const uint32_t tt = Lp % a.tok_tiles, rg = Lp / a.tok_tiles;
    const uint32_t tok0 = tt * a.tok_tile;
    const uint32_t ntile = a.n_tok - tok0 < a.tok_tile ? a.n_tok - tok0 : a.tok_tile;

    const uint32_t lane = threadIdx.x & 63u, n = lane & 15u, kg = lane >> 4;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t S = a.splits, R = a.waves / S, rt = wv % R, ks = wv / R;
    if constexpr (FFN) pi = rt / (R / 2);
    const FewPart &P = a.p[pi];
    const uint32_t row0 = FFN ? rg * 32 + (rt % (R / 2)) * 16 : (rg * R + rt) * 16;

    FewAct A;
    A.ntp = (ntile + 3u) & ~3u;
    A.stride = a.kpad + kRowPad;
    A.fsc = reinterpret_cast<float *>(smem);
    A.fx = A.fsc + (a.kpad / 32) * A.ntp;
    A.codes = reinterpret_cast<uint8_t *>(A.fx + (TYPE == AH_GGML_Q4_K ? a.kpad / 32 : TYPE == AH_GGML_Q2_K ? a.kpad / 16 : 0u) * A.ntp);

    uint8_t *const slot = A.codes + ntile * A.stride + wv * Unit<TYPE>::slot;

    const uint32_t nu = (a.n_in + Unit<TYPE>::k - 1) / Unit<TYPE>::k;
    FewWave<TYPE, NT> W;
    W.rs = ah_rsrc(P.w, P.w_bytes);
    W.rb = (row0 + n < P.n_out ? row0 + n : 0u) * P.row_bytes;
    W.n_in = a.n_in;
    W.n = n;
    W.kg = kg;
    const uint32_t u0 = nu * ks / S;
    W.u1 = nu * (ks + 1) / S;
    W.plan(row0, P.n_out, P.row_bytes, lane);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        // tokens past the tile read one inside it; their sums are never stored
        W.tok[j] = 16 * j + n < ntile ? 16 * j + n : ntile - 1;
        W.grp[j] = 16 * j + 4 * kg < A.ntp ? 16 * j + 4 * kg : 0u;
#pragma unroll
        for (int r = 0; r < 4; ++r) W.acc[j][r] = 0.0f;
    }
    if (u0 < W.u1) W.load(u0);
    if (a.src == AH_SRC_F32) stage_f32<TYPE>(a, A, tok0, ntile);
    else if (((uint32_t)reinterpret_cast<uintptr_t>(a.x) | a.pitch) & 3u) stage_codes<TYPE, true>(a, A, tok0, ntile);
    else stage_codes<TYPE, false>(a, A, tok0, ntile);
    ah_lds_barrier();
    for (uint32_t u = u0; u < W.u1; ++u) {
        W.stage(slot, lane);
        if (u + 1 < W.u1) W.load(u + 1);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's LDS stores have landed
        __builtin_amdgcn_wave_barrier();
        W.compute(A, slot, u);
        __builtin_amdgcn_wave_barrier();  // all lanes are done reading the slot before it is refilled
    }
    // the splits' sums meet in LDS, [ks][row tile][token][row], over the activations
    ah_lds_barrier();
    float *const red = reinterpret_cast<float *>(smem);
    constexpr uint32_t kTile = 256 * NT;  // sums of one row tile
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(ks * R + rt) * kTile + (16 * j + 4 * kg + r) * 16 + n] = W.acc[j][r];
    ah_lds_barrier();
    if constexpr (!FFN) {
        for (uint32_t i = threadIdx.x; i < R * kTile; i += blockDim.x) {
            const uint32_t tl = (i % kTile) / 16, row = (rg * R + i / kTile) * 16 + (i & 15u);
            float s = 0.0f;
            for (uint32_t k = 0; k < S; ++k) s += red[k * R * kTile + i];
            if (tl >= ntile || row >= P.n_out) continue;
            const uint64_t e = (uint64_t)(tok0 + tl) * P.n_out + row;
            P.y[e] = s;
            if (const uint32_t oc = ah_out_code(s)) ah_record(a.status, ah_out_key(P.key0 + e, oc));
        }
    } else {
        // one hidden value per thread, 32 lanes per token: its gate and up sums, then the SwiGLU and the
        // hidden quantizer.  Refusals in the reference FFN's order (chart/ffn.rs:1712-1720), keyed as
        // the other prefill forms key them.
        const uint32_t n_ff = P.n_out, nbh = (n_ff + 31) / 32;
        const uint64_t NF = (uint64_t)a.n_tok * n_ff;
        for (uint32_t i = threadIdx.x; i < 32 * ((ntile + 1) & ~1u); i += blockDim.x) {  // whole waves
            const uint32_t tl = i / 32, l = i & 31u, k = 32 * rg + l;
            const bool live = tl < ntile && k < n_ff;
            const uint64_t t = (uint64_t)tok0 + tl, e = t * n_ff + k;
            const uint32_t at = (l / 16) * kTile + (tl < ntile ? tl : 0u) * 16 + (l & 15u);
            float g = 0.0f, u = 0.0f;
            for (uint32_t s = 0; s < S; ++s) {
                g += red[s * R * kTile + at];
                u += red[(s * R + R / 2) * kTile + at];
            }
            if (live) {
                if (a.gy) a.gy[e] = g;
                if (a.uy) a.uy[e] = u;
                if (const uint32_t oc = ah_out_code(g)) ah_record(a.status, ah_out_key(e, oc));
                if (const uint32_t oc = ah_out_code(u)) ah_record(a.status, ah_out_key(NF + e, oc));
            }
            const HiddenQ q = swiglu_quant32(__builtin_bit_cast(uint32_t, g), __builtin_bit_cast(uint32_t, u), live);
            if (q.err) ah_record(a.status, ah_out_key(2 * NF + e, (uint32_t)q.err));
            if (live) a.h_codes[e] = (int8_t)q.code;
            if (live && l == 0) {
                if (q.bad_block) ah_record(a.status, ah_out_key(3 * NF + t * nbh + rg, 7u));
                a.h_scales[t * nbh + rg] = (int64_t)q.scale;
            }
        }
    }
}

template <int NT, bool FFN>
const void *few_fn(uint32_t type) {
    switch (type) {
    case AH_GGML_Q8_0: return reinterpret_cast<const void *>(&gemm_few_kernel<AH_GGML_Q8_0, NT, FFN>);
    case AH_GGML_Q5_0: return reinterpret_cast<const void *>(&gemm_few_kernel<AH_GGML_Q5_0, NT, FFN>);
    case AH_GGML_Q2_K: return reinterpret_cast<const void *>(&gemm_few_kernel<AH_GGML_Q2_K, NT, FFN>);
    case AH_GGML_Q3_K: return reinterpret_cast<const void *>(&gemm_few_kernel<AH_GGML_Q3_K, NT, FFN>);
    case AH_GGML_Q4_K: return reinterpret_cast<const void *>(&gemm_few_kernel<AH_GGML_Q4_K, NT, FFN>);
    case AH_GGML_Q6_K: return reinterpret_cast<const void *>(&gemm_few_kernel<AH_GGML_Q6_K, NT, FFN>);
    default: return nullptr;
    }
}
const void *few_fn(uint32_t type, uint32_t nt, bool ffn) {
    return ffn ? (nt == 1 ? few_fn<1, true>(type) : few_fn<2, true>(type))
               : (nt == 1 ? few_fn<1, false>(type) : few_fn<2, false>(type));
}

}  // namespace

// LDS of a workgroup of `tok` tokens: the quantized activations, or the splits' sums over them.
size_t ah_few_lds_bytes(uint32_t type, uint32_t kpad, uint32_t tok, uint32_t waves) {
    const size_t ntp = (tok + 3u) & ~3u;
    const size_t fx = type == AH_GGML_Q4_K ? kpad / 32 : type == AH_GGML_Q2_K ? kpad / 16 : 0;
    const size_t act = (kpad / 32 + fx) * ntp * 4 + (size_t)tok * (kpad + kRowPad) + (size_t)waves * slot_of(type) + 16;
    const size_t red = (size_t)waves * 256 * (tok > 16 ? 2 : 1) * 4;
    return act > red ? act : red;
}

// Waves along K of a row tile: three units each (the later two stream in while the wave computes),
// at most kFewMaxWaves.  More, shorter waves measured no faster (896 x 896 6.2 us either way) and
// fewer leave a deep product to few CUs.  The choice depends on the part alone, so that a grouped
// part, and a gate or up projection with the SwiGLU epilogue, is what its single call computes.
uint32_t ah_few_splits(uint32_t type, uint32_t n_in) {
    const uint32_t nu = (n_in + unit_k_of(type) - 1) / unit_k_of(type);
    uint32_t s = (nu + 2) / 3;
    s = s < 1 ? 1 : s > kFewMaxWaves ? kFewMaxWaves : s;
    const uint32_t per = (nu + s - 1) / s;
    return per ? (nu + per - 1) / per : 1;  // the same longest wave with the fewest of them
}

// us of `wgs` workgroups of `tok` tokens past a launch's fixed time, where they take more than one
// round over the CUs (0: one round, in which the route was the faster one at every size measured):
// 5.1 a round, and for each workgroup a CU runs the staging of its tokens and the folds of its
// units.  A CU holds the workgroups that fit its LDS and the waves that fit its registers: 24 at 80
// VGPRs, 20 at 87 (Q2_K and Q6_K), 16 with two operand tiles.  ah_abi.cpp compares it with the tile
// GEMM's.
double ah_few_cost(uint32_t type, uint32_t n_in, uint32_t kpad, uint32_t tok, uint32_t splits, uint32_t waves, size_t wgs, uint32_t cus) {
    const size_t by_lds = 160 * 1024 / ah_few_lds_bytes(type, kpad, tok, waves), by_waves = (tok > 16 ? 16 : type == AH_GGML_Q2_K || type == AH_GGML_Q6_K ? 20 : 24) / waves;
    const size_t held = by_lds < by_waves ? by_lds : by_waves, per_round = cus * (held ? held : 1);
    const size_t rounds = (wgs + per_round - 1) / per_round;
    if (rounds <= 1) return 0.0;
    const uint32_t nu = (n_in + unit_k_of(type) - 1) / unit_k_of(type), per = (nu + splits - 1) / splits;
    const double fold = type == AH_GGML_Q4_K ? 1.5 : type == AH_GGML_Q2_K ? 1.13 : type == AH_GGML_Q6_K ? 0.75 : type == AH_GGML_Q3_K ? 0.32 : 0.46;
    return 5.1 * (double)rounds + (double)((wgs + cus - 1) / cus) * (0.24e-4 * tok * kpad + fold * (waves * per * (tok > 16 ? 2 : 1)) / 16.0);
}

hipError_t ah_few_init_attrs() {
    for (uint32_t t : {AH_GGML_Q8_0, AH_GGML_Q5_0, AH_GGML_Q2_K, AH_GGML_Q3_K, AH_GGML_Q4_K, AH_GGML_Q6_K})
        for (uint32_t nt = 1; nt <= 2; ++nt)
            for (int f = 0; f < 2; ++f) {
                const hipError_t e = hipFuncSetAttribute(few_fn(t, nt, f != 0), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
                if (e != hipSuccess) return e;
            }
    return hipSuccess;
}

// Fills each part's wg_begin and the workgroup count, then launches.  FFN: parts {gate, up} of one
// type and shape, one workgroup per hidden 32-block and token tile.
hipError_t ah_launch_few(uint32_t type, FewArgs &a, bool ffn, hipStream_t stream) {
    const uint32_t nt = a.tok_tile > 16 ? 2u : 1u;
    const void *f = few_fn(type, nt, ffn);
    if (!f || a.n_parts == 0 || a.n_parts > kFewMaxParts || a.tok_tile == 0 || a.tok_tile > 32 || a.splits == 0 ||
        a.waves > kFewMaxWaves || a.waves == 0 || a.waves % a.splits || (ffn && (a.n_parts != 2 || a.waves != 4 * a.splits)))
        return hipErrorInvalidValue;
    a.tok_tiles = (a.n_tok + a.tok_tile - 1) / a.tok_tile;
    const uint32_t rows = 16 * (a.waves / a.splits);
    uint32_t wg = 0;
    for (uint32_t i = 0; i < a.n_parts; ++i) {
        a.p[i].wg_begin = wg;
        if (!ffn || i == 0) wg += (a.p[i].n_out + (ffn ? 32 : rows) - 1) / (ffn ? 32 : rows) * a.tok_tiles;
    }
    a.n_wg = wg;
    if (wg == 0) return hipSuccess;
    const uint32_t tok = a.n_tok < a.tok_tile ? a.n_tok : a.tok_tile;
    void *args[] = {&a};
    return hipLaunchKernel(f, dim3((wg + 7) / 8 * 8), dim3(64 * a.waves), args, ah_few_lds_bytes(type, a.kpad, tok, a.waves), stream);
}
