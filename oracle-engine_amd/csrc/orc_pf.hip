// Prefill GEMM on the matrix cores (gfx950): many-token calls (the batched
// prompt pass of Model::forward_prefill, core/model.cpp:510-674) on Q4_K,
// Q6_K, Q8_0 (GGUF blocks or regrouped), Q4_0, F16 and BF16 weights, with the
// RMSNorm prologue and the bias / residual / SwiGLU epilogues.
//
// Two launches per call (one k_pf_split for all weight types of a call, one
// k_pf per run of segments of one type):
//  * k_pf_split writes the activations once, split exactly as the MFMA reads
//    them: x' = x times the norm weight times a power of two per (token,
//    256 values), hi = fp16(x'), lo = fp16(x' - hi) (~22 bits; BF16 weights:
//    three bf16 pieces, 24 bits, no scaling), in whole 1 KB fragments, with
//    the powers, the sums of x^2 for the norm and, for Q4_K, the sums over
//    each 32-value sub-block.
//  * k_pf streams those fragments through the LDS while every wave decodes
//    its own weight rows straight from the GGUF blocks into B operands:
//    products of fp16 halves with exact weight codes are exact in fp32.
// Before, every workgroup of the GEMM split its tokens' activations itself
// (rows / 128 times over, more vector work than the products), and calls
// below 256 tokens re-read and re-decoded the weights for each block of 5-16
// tokens. Measured (MI355X, us before -> after): 7B gate+up Q6_K 37888 x 3584
// at 1023 tokens 1790 -> 891 (3.1e14 flop/s; at three MFMAs per product 74% of
// what the card's bf16 library product reaches), at 127 tokens 741 -> 171;
// 3B gate+up Q4_K 16384 x 3072 484 -> 304 and 178 -> 60; F16 16384 x 2048
// 3168 -> 204 and 411 -> 45; 0.5B gate+up Q8_0 9728 x 896 236 -> 87. Error
// against 64 bits: Q6_K 3584 values 1.1e-7 of the result's rms (1.2e-7 and
// 1.6e-7 before), Q4_K 1.4e-7 (2.0e-7, 3.3e-7), Q8_0 1.0e-7 (3.9e-7). Calls of
// Q4_0, F16 and of 24 to 255 tokens of Q8_0 had fp32 activations before: over
// 1B-shape blocks of 24 to 600 tokens Q4_0 2.2e-7 -> 1.0e-7, F16 1.4e-7 ->
// 1.2e-7, Q8_0 3.9e-7 -> 1.1e-7 per product, the sums outweighing the two bits.
// A value more than 2^17 below the largest of its token's 256 keeps fewer bits
// than the others (14 at 2^24), as in the verify kernels of the K-quants.
// What bounds k_pf: weight rows are read 32 bytes per lane pair (one cache
// line per row and load: with all lanes on one row 7B gate+up took a third
// less), the LDS reads of the fragments (1 KB per MFMA pair) and, at few
// tokens, the latency of a stage. GGUF Q8_0 and Q4_0 rows join their two block
// scales as they are loaded, so a stage of theirs waits for the next one's
// loads before its products (4.8 us a superblock of a lone chain against 2.7).
//
// The workspace between the two launches belongs to the library (one per
// device, allocated by orc_init): calls take it in turn, ordered across
// streams by an event, so prefill calls on two streams do not overlap, and on a
// stream the library did not create each is followed by an event (4.4 us). A call whose stream is being captured does not use it
// (a graph could replay while another stream uses the workspace) and takes
// the kernels that stage x themselves (orc_mmq.hip, orc_gemm.hip).
#include "orc_gemm.hpp"

#include <algorithm>
#include <mutex>
#include <string>

namespace orc {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));

typedef const __attribute__((address_space(1))) u32x4_u* g16p;
typedef const __attribute__((address_space(1))) u32x2_u* g8p;
typedef const __attribute__((address_space(1))) u32_u* g4p;
typedef const __attribute__((address_space(1))) u16_u* g2p;
typedef const __attribute__((address_space(1))) float* gfp;
typedef __attribute__((address_space(1))) float* gwp;
__device__ __forceinline__ u32x4 ldg16(const uint8_t* p) { return *(g16p)p; }
__device__ __forceinline__ u32x2 ldg8(const uint8_t* p) { return *(g8p)p; }
__device__ __forceinline__ uint32_t ldg4(const uint8_t* p) { return *(g4p)p; }
__device__ __forceinline__ uint32_t ldg2(const uint8_t* p) { return *(g2p)p; }

__device__ __forceinline__ h2v as_h2(uint32_t v) { return __builtin_bit_cast(h2v, v); }
__device__ __forceinline__ uint32_t as_u32(h2v v) { return __builtin_bit_cast(uint32_t, v); }

// A constant kept in a register: (x & mask) | magic is then one v_and_or_b32,
// which takes at most one literal.
__device__ __forceinline__ uint32_t vconst(uint32_t c) {
    asm("" : "+v"(c));
    return c;
}

// ── layout ───────────────────────────────────────────────────────────────────
// Activations in groups of 32 tokens, K in stages of 64 values (a whole number
// of 128-value units, zero beyond n_in). A fragment is the A operand of one
// v_mfma_f32_32x32x16: lane l holds token l % 32, eight values of the half
// h = l / 32. Step s = 2 b + a of a stage covers block b (32 values): half h,
// values 32 b + 16 h + 8 a + 0 .. 7, so that a lane's two steps of a block are
// 16 consecutive codes of its weight row. Inside the eight, quantized types
// take the order 0 2 1 3 4 6 5 7 in which bytes unpack into fp16 pairs.
// Odd blocks (b = 1) are stored negated and their products subtracted: the
// matrix cores round their sums toward minus infinity, a bias that would grow
// with the row's length (mean error -1.5e-7 of a result's rms at 18944 values,
// 2.4e-7 in all); with half the sums negated it cancels.
// frag(group, stage, step, piece) = ((group * stages + stage) * 4 + step) *
// pieces + piece, 1 KB each.
constexpr int kFragBytes = 1024, kStage = 64, kSuper = 256;

struct PfWork {          // where one call's split activations live
    uint8_t* frag;       // fragments
    float* es;           // [group][superblock][32 tokens]: 2^-e
    float* ss;           // the same shape: sums of x^2
    uint8_t* sums;       // Q4_K: [group][superblock][2] fragments of sub-block sums
    int stages, supers;  // per token group
};

struct PfSplit {
    PfWork w;
    const float *x, *norm_w;
    int ldx, n_tok, n_in;
};

// PL pieces per value: 2 (fp16 hi, lo) or 3 (bf16). PERM: byte-unpack order.
// One workgroup per (256 values, 32 tokens): wave w one 64-value stage; lane:
// one token, 16 values of each of the stage's two blocks. Reads each x once
// and writes whole fragments (64 lanes x 16 bytes); bound by memory.
template <int PL, bool PERM, bool SUMS>
__global__ __launch_bounds__(256) void k_pf_split(PfSplit p) {
    __shared__ float smx[4][32], sss[4][32], ssum[8][32];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, tl = lane & 31, h = lane >> 5;
    const int sb = blockIdx.x, grp = blockIdx.y, st = 4 * sb + w, tok = grp * 32 + tl;
    const bool in = tok < p.n_tok;
    const float* xr = p.x + (size_t)(in ? tok : 0) * p.ldx;
    float v[2][16], gw[2][16];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int k0 = st * kStage + 32 * b + 16 * h;
        const bool ok = in && k0 < p.n_in;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 a = ok ? *(const float4*)(xr + k0 + 4 * j) : make_float4(0.f, 0.f, 0.f, 0.f);
            v[b][4 * j] = a.x, v[b][4 * j + 1] = a.y, v[b][4 * j + 2] = a.z, v[b][4 * j + 3] = a.w;
            if (p.norm_w) {
                const float4 g = k0 < p.n_in ? *(const float4*)(p.norm_w + k0 + 4 * j) : make_float4(0.f, 0.f, 0.f, 0.f);
                gw[b][4 * j] = g.x, gw[b][4 * j + 1] = g.y, gw[b][4 * j + 2] = g.z, gw[b][4 * j + 3] = g.w;
            }
        }
    }
    float ssq = 0.f, mx = 0.f, s32[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            ssq = __builtin_fmaf(v[b][i], v[b][i], ssq);
            if (p.norm_w) v[b][i] *= gw[b][i];
            const float a = fabsf(v[b][i]);
            mx = fmaxf(mx, a <= 3.4028234e38f ? a : 0.f);  // infinities and NaN set no scale
        }
        if constexpr (SUMS) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < 16; i += 4) s += (v[b][i] + v[b][i + 1]) + (v[b][i + 2] + v[b][i + 3]);
            s32[b] = s + __shfl_xor(s, 32, 64);
        }
    }
    ssq += __shfl_xor(ssq, 32, 64);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (h == 0) {
        smx[w][tl] = mx;
        sss[w][tl] = ssq;
        if constexpr (SUMS) ssum[2 * w][tl] = s32[0], ssum[2 * w + 1][tl] = s32[1];
    }
    __syncthreads();
    float up = 1.f, es = 1.f;
    if constexpr (PL == 2) {  // max |x'| below 2^14
        mx = fmaxf(fmaxf(smx[0][tl], smx[1][tl]), fmaxf(smx[2][tl], smx[3][tl]));
        int e2 = 0;
        if (mx > 0.f) {
            int ex;
            (void)frexpf(mx, &ex);  // mx < 2^ex
            e2 = min(14 - ex, 120);
        }
        up = ldexpf(1.f, e2);
        es = ldexpf(1.f, -e2);
    }
    const size_t so = ((size_t)grp * p.w.supers + sb) * 32 + tl;
    if (tid < 32) {
        p.w.es[so] = es;
        p.w.ss[so] = (sss[0][tl] + sss[1][tl]) + (sss[2][tl] + sss[3][tl]);
    }
    if (st < p.w.stages) {
        uint8_t* dst = p.w.frag + ((size_t)grp * p.w.stages + st) * (4 * PL * kFragBytes) + lane * 16;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int b = s >> 1, i0 = 8 * (s & 1);
            const float ub = b ? -up : up;  // odd blocks negated
            uint32_t o[PL][4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                // positions 2q, 2q + 1 of the eight
                const int ea = PERM ? (q & 2) * 2 + (q & 1) : 2 * q, eb = PERM ? ea + 2 : ea + 1;
                if constexpr (PL == 2) {
                    const f2v a = {v[b][i0 + ea] * ub, v[b][i0 + eb] * ub};
                    const h2v hi = __builtin_convertvector(a, h2v);
                    f2v r = {a.x - (float)hi.x, a.y - (float)hi.y};
                    if (!(fabsf(a.x) <= 3.4028234e38f)) r.x = 0.f;  // an infinity or NaN is its hi half alone
                    if (!(fabsf(a.y) <= 3.4028234e38f)) r.y = 0.f;
                    o[0][q] = as_u32(hi);
                    o[1][q] = as_u32(__builtin_convertvector(r, h2v));
                } else {
                    float a[2] = {v[b][i0 + ea] * ub, v[b][i0 + eb] * ub};
#pragma unroll
                    for (int pl = 0; pl < PL; ++pl) {
                        uint32_t bits = 0;
#pragma unroll
                        for (int z = 0; z < 2; ++z) {
                            const __bf16 c = (__bf16)a[z];
                            bits |= (uint32_t)__builtin_bit_cast(uint16_t, c) << (16 * z);
                            const float f = (float)c;
                            a[z] = fabsf(f) <= 3.4028234e38f ? a[z] - f : 0.f;
                        }
                        o[pl][q] = bits;
                    }
                }
            }
#pragma unroll
            for (int pl = 0; pl < PL; ++pl)
                *(u32x4*)(dst + (s * PL + pl) * kFragBytes) = u32x4{o[pl][0], o[pl][1], o[pl][2], o[pl][3]};
        }
    }
    if constexpr (SUMS) {
        // sums of x' over the eight sub-blocks, in three exact fp16 pieces
        // (times 2^-6, so they stay in range): fragment 0 holds hi | mid,
        // fragment 1 lo | 0 in its two halves of K
        if (w == 0) {
            h8v f0, f1;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float s = ssum[j][tl] * up * 0.015625f;
                const bool fin = fabsf(s) <= 3.4028234e38f;
                const _Float16 a = (_Float16)s;
                const float r = fin ? s - (float)a : 0.f;
                const _Float16 m = (_Float16)r;
                const _Float16 l = (_Float16)(r - (float)m);
                f0[j] = h ? m : a;
                f1[j] = h ? (_Float16)0.f : l;
            }
            uint8_t* d = p.w.sums + ((size_t)grp * p.w.supers + sb) * (2 * kFragBytes) + lane * 16;
            *(h8v*)d = f0;
            *(h8v*)(d + kFragBytes) = f1;
        }
    }
}

// ── weight rows ──────────────────────────────────────────────────────────────
// A lane's share of its row for GR stages (a granule): the codes of its half
// h of every 32-value block. block(b) prepares block b (0 .. 2 GR - 1) of the
// granule, step(a) gives the B operand of the block's step a, scale() what
// the block's products are multiplied by.
template <int QT> struct PfRow;

// four code bytes as fp16 1024 + code in two words: bytes 0, 2 | bytes 1, 3
__device__ __forceinline__ void unpack4(uint32_t w, uint32_t mk, uint32_t mg, uint32_t& r0, uint32_t& r1) {
    r0 = (w & mk) | mg;
    r1 = ((w >> 8) & mk) | mg;
}

template <> struct PfRow<ORC_Q4_K> {
    // core/gguf_parser.cpp:1096-1121: stage j of a superblock is its chunk of
    // 32 code bytes (block 0: low nibbles, block 1: high nibbles), this
    // lane's 16 of them one load. A value is d sc (q - 8) + (8 d sc - dmin m):
    // sc (q - 8) is exact in fp16, and the second part meets only the
    // sub-block's sum of x. Centred codes keep the products' sum near the
    // result's size (with q in 0 .. 15 it is twice as large, and so is its
    // rounding).
    static constexpr int GR = 1, PL = 2;
    static constexpr bool SPLIT = false, MINS = true, BF = false;
    u32x4 hdr, q;
    h2v scv, off;
    __device__ __forceinline__ void load(const uint8_t* row, int st, int h, int) {
        const uint8_t* blk = row + (size_t)(st >> 2) * 144;
        hdr = ldg16(blk);
        q = ldg16(blk + 16 + 32 * (st & 3) + 16 * h);
    }
    __device__ __forceinline__ void block(int b, int st, int) {
        uint32_t sc, mn;
        q4k_scale_min(2 * (st & 3) + b, hdr.y, hdr.z, hdr.w, sc, mn);
        const float f = (float)sc;
        // nibbles at bit 4 of each byte: (1024 + 16 q) (sc / 16) - 72 sc = sc (q - 8), exact
        const _Float16 s = (_Float16)(f * 0.0625f), o = (_Float16)(f * -72.f);
        scv = h2v{s, s};
        off = h2v{o, o};
    }
    __device__ __forceinline__ void step(int b, int a, h8v& hi, h8v&) const {
        const uint32_t mk = 0x00F000F0u, mg = vconst(0x64006400u);
        const uint32_t w0 = a ? q.z : q.x, w1 = a ? q.w : q.y;
        const uint32_t t[4] = {((b ? w0 : w0 << 4) & mk) | mg, ((w0 >> (b ? 8 : 4)) & mk) | mg,
                               ((b ? w1 : w1 << 4) & mk) | mg, ((w1 >> (b ? 8 : 4)) & mk) | mg};
        u32x4 r;
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] = as_u32(__builtin_elementwise_fma(as_h2(t[k]), scv, off));
        hi = __builtin_bit_cast(h8v, r);
    }
    __device__ __forceinline__ float scale() const { return h2f(hdr.x & 0xFFFFu); }
    __device__ __forceinline__ float dmin() const { return h2f(hdr.x >> 16); }
    // the superblock's eight scales and minimums as fp16
    __device__ __forceinline__ void scales(h8v& sc8, h8v& mn8) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            uint32_t sc, mn;
            q4k_scale_min(j, hdr.y, hdr.z, hdr.w, sc, mn);
            sc8[j] = (_Float16)(float)sc;
            mn8[j] = (_Float16)(float)mn;
        }
    }
};

template <> struct PfRow<ORC_Q6_K> {
    // core/gguf_parser.cpp:1124-1154: a granule is half a superblock (128
    // values, four blocks); sc (q - 32) in an fp16 half and its exact
    // remainder (|lo| <= 1; see mmq_core_q6k)
    static constexpr int GR = 2, PL = 2;
    static constexpr bool SPLIT = true, MINS = false, BF = false;
    u32x4 la, lb, qh;
    u32x2 sc;
    uint32_t dh;
    h2v sc2;
    __device__ __forceinline__ void load(const uint8_t* row, int st, int h, int) {
        const uint8_t* blk = row + (size_t)(st >> 2) * 210;
        const int hh = (st >> 1) & 1;
        la = ldg16(blk + 64 * hh + 16 * h);
        lb = ldg16(blk + 64 * hh + 32 + 16 * h);
        qh = ldg16(blk + 128 + 32 * hh + 16 * h);
        sc = ldg8(blk + 192 + 8 * hh);
        dh = ldg2(blk + 208);
    }
    __device__ __forceinline__ void block(int b, int, int h) {
        const uint32_t sw = b < 2 ? sc.x : sc.y;
        const _Float16 s = (_Float16)(float)(int8_t)((sw >> (16 * (b & 1) + 8 * h)) & 0xFFu);
        sc2 = h2v{s, s};
    }
    __device__ __forceinline__ void step(int b, int a, h8v& hi, h8v& lo) const {
        const u32x4 l = (b & 1) ? lb : la;
        const h2v off{(_Float16)-1056.f, (_Float16)-1056.f};  // 1024 + 32
        const uint32_t mg = vconst(0x64646464u);
        u32x4 rh, rl;
#pragma unroll
        for (int z = 0; z < 2; ++z) {
            const uint32_t lw = z ? (a ? l.w : l.y) : (a ? l.z : l.x);
            const uint32_t hw = z ? (a ? qh.w : qh.y) : (a ? qh.z : qh.x);
            const uint32_t hb = (b < 2 ? hw << (4 - 2 * b) : hw >> (2 * b - 4)) & 0x30303030u;
            const uint32_t q = ((b >> 1 ? lw >> 4 : lw) & 0x0F0F0F0Fu) | hb;
            const uint32_t r[2] = {__builtin_amdgcn_perm(mg, q, 0x04020400u), __builtin_amdgcn_perm(mg, q, 0x04030401u)};
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const h2v v = as_h2(r[k]) + off;  // q - 32, exact
                const h2v t = v * sc2;
                rh[2 * z + k] = as_u32(t);
                rl[2 * z + k] = as_u32(__builtin_elementwise_fma(v, sc2, -t));
            }
        }
        hi = __builtin_bit_cast(h8v, rh);
        lo = __builtin_bit_cast(h8v, rl);
    }
    __device__ __forceinline__ float scale() const { return h2f(dh); }
};

// Q8_0 (core/gguf_parser.cpp:1073-1082), GGUF blocks or regrouped: a stage is
// two blocks; the codes are exact in fp16, the block scale is not folded in
// (an 11-bit scale times an 8-bit code would be rounded) but applied to the
// block's products
template <bool X8> struct PfRowQ8 {
    static constexpr int GR = 1, PL = 2;
    static constexpr bool SPLIT = false, MINS = false, BF = false;
    u32x4 q[2];
    uint32_t dh;
    float db;
    __device__ __forceinline__ void load(const uint8_t* row, int st, int h, int n_blk) {
        if constexpr (X8) {
            const uint8_t* g = row + (size_t)(st >> 2) * 272;
            const int b0 = 2 * (st & 3);
            dh = ldg4(g + 2 * b0);
#pragma unroll
            for (int b = 0; b < 2; ++b) q[b] = ldg16(g + 16 + 32 * (b0 + b) + 16 * h);
        } else {
            uint32_t s[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int blk = min(2 * st + b, n_blk - 1);  // past the row's end: x is zero
                const uint8_t* g = row + (size_t)blk * 34;
                s[b] = ldg2(g);
                q[b] = ldg16(g + 2 + 16 * h);
            }
            dh = s[0] | (s[1] << 16);
        }
    }
    __device__ __forceinline__ void block(int b, int, int) { db = h2f(b ? dh >> 16 : dh & 0xFFFFu); }
    __device__ __forceinline__ void step(int b, int a, h8v& hi, h8v&) const {
        // code + 128 in the low byte of fp16 1024 + b, then 1152 comes off
        const uint32_t m = 0x00FF00FFu, mg = vconst(0x64006400u);
        const h2v off{(_Float16)-1152.f, (_Float16)-1152.f};
        u32x4 r;
        uint32_t t[4];
        unpack4((a ? q[b].z : q[b].x) ^ 0x80808080u, m, mg, t[0], t[1]);
        unpack4((a ? q[b].w : q[b].y) ^ 0x80808080u, m, mg, t[2], t[3]);
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] = as_u32(as_h2(t[k]) + off);
        hi = __builtin_bit_cast(h8v, r);
    }
    __device__ __forceinline__ float scale() const { return db; }
};
template <> struct PfRow<ORC_Q8_0> : PfRowQ8<false> {};
template <> struct PfRow<ORC_Q8_0_X8> : PfRowQ8<true> {};

// Q4_0 (core/gguf_parser.cpp:1058-1070): half h of a block is one nibble of
// all 16 code bytes
template <> struct PfRow<ORC_Q4_0> {
    static constexpr int GR = 1, PL = 2;
    static constexpr bool SPLIT = false, MINS = false, BF = false;
    u32x4 q[2];
    uint32_t dh;
    int sh;
    float db;
    __device__ __forceinline__ void load(const uint8_t* row, int st, int h, int n_blk) {
        uint32_t s[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int blk = min(2 * st + b, n_blk - 1);
            const uint8_t* g = row + (size_t)blk * 18;
            s[b] = ldg2(g);
            q[b] = ldg16(g + 2);
        }
        dh = s[0] | (s[1] << 16);
        sh = 4 * h;
    }
    __device__ __forceinline__ void block(int b, int, int) { db = h2f(b ? dh >> 16 : dh & 0xFFFFu); }
    __device__ __forceinline__ void step(int b, int a, h8v& hi, h8v&) const {
        const uint32_t m = 0x000F000Fu, mg = vconst(0x64006400u);
        const h2v off{(_Float16)-1032.f, (_Float16)-1032.f};
        u32x4 r;
        uint32_t t[4];
        unpack4((a ? q[b].z : q[b].x) >> sh, m, mg, t[0], t[1]);
        unpack4((a ? q[b].w : q[b].y) >> sh, m, mg, t[2], t[3]);
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] = as_u32(as_h2(t[k]) + off);
        hi = __builtin_bit_cast(h8v, r);
    }
    __device__ __forceinline__ float scale() const { return db; }
};

// F16 / BF16 rows: the values themselves
template <bool B16> struct PfRowDense {
    static constexpr int GR = 1, PL = B16 ? 3 : 2;
    static constexpr bool SPLIT = false, MINS = false, BF = B16;
    u32x4 q[2][2];
    __device__ __forceinline__ void load(const uint8_t* row, int st, int h, int n_blk) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int blk = min(2 * st + b, n_blk - 1);
#pragma unroll
            for (int a = 0; a < 2; ++a) q[b][a] = ldg16(row + (size_t)blk * 64 + 32 * h + 16 * a);
        }
    }
    __device__ __forceinline__ void block(int, int, int) {}
    __device__ __forceinline__ void step(int b, int a, h8v& hi, h8v&) const { hi = __builtin_bit_cast(h8v, q[b][a]); }
    __device__ __forceinline__ float scale() const { return 1.f; }
};
template <> struct PfRow<ORC_F16> : PfRowDense<false> {};
template <> struct PfRow<ORC_BF16> : PfRowDense<true> {};

template <bool BF> __device__ __forceinline__ f16v mfma(h8v a, h8v b, f16v c) {
    if constexpr (BF)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8v, a), __builtin_bit_cast(b8v, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

template <class T> __device__ __forceinline__ T* spin(T* p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (T*)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ int seg_of(int j, int n_seg, int r0, int r1, int& jj) {
    const bool s1 = n_seg > 1 && j >= r0, s2 = n_seg > 2 && j >= r0 + r1;
    jj = s2 ? j - r0 - r1 : (s1 ? j - r0 : j);
    return s2 ? 2 : (s1 ? 1 : 0);
}
template <class T> __device__ __forceinline__ T* pick3(int s, T* a, T* b, T* c) { return s == 2 ? c : (s == 1 ? b : a); }

// 1 / rms of a token: its superblocks' sums of x^2 in order
__device__ __forceinline__ float pf_inv_rms(const PfWork& wk, int grp, int tl, int n_in, float eps) {
    const float* sp = wk.ss + (size_t)grp * wk.supers * 32 + tl;
    float ss = 0.f;
    for (int i = 0; i < wk.supers; ++i) ss += *(gfp)(sp + 32 * i);
    return 1.f / sqrtf(ss / (float)n_in + eps);
}
// one output value: v (SwiGLU: gate v, up u), bias 0 without one
__device__ __forceinline__ void pf_write(const QmvParams& p, float* y, float v, float u, float bias) {
    if (p.epi == ORC_EPI_SWIGLU) *(gwp)y = (v / (1.f + expf(-v))) * u;
    else if (p.epi == ORC_EPI_ACCUM) *(gwp)y += v + bias;
    else *(gwp)y = v + bias;
}

// ── the GEMM ─────────────────────────────────────────────────────────────────
// RW waves; a wave computes 32 rows by TT tiles of 32 tokens (TT = 4: a
// workgroup's 128 rows x 128 tokens). SwiGLU: a wave's rows are 16 gate rows
// and their 16 up rows. blockIdx.z takes one of gridDim.z contiguous ranges of
// superblocks; with more than one the raw sums go to `part` and k_pf_sum adds
// them up and does the epilogue.
// A (token, row) sum: per 32-value block one chain of products, the small
// pieces first; the blocks' chains times their scales in order per 256
// values; those times 2^-e in order over the row. Three levels keep the
// rounding of a long row near that of the vector kernels' lane-wise sums.
// The order is the same for every tile shape and every token count: a result
// depends on nothing else in the launch but the number of ranges.
template <int QT, int RW, int TT>
__global__ __launch_bounds__(64 * RW) __attribute__((amdgpu_waves_per_eu(2))) void k_pf(QmvParams p, PfWork wk,
                                                                                          float* part) {
    using Row = PfRow<QT>;
    constexpr int PL = Row::PL, GR = Row::GR, NTH = 64 * RW, BT = 32 * TT;
    constexpr int kGrpStage = 4 * PL * kFragBytes;                  // bytes of a token group's stage
    constexpr int kStageBytes = TT * kGrpStage;                     // of the workgroup's
    constexpr int NC = kStageBytes / 16 / NTH;                      // fragments a wave copies per stage
    static_assert(kStageBytes % (16 * NTH) == 0, "whole fragments");
    static_assert(BT <= NTH, "one thread per token");
    extern __shared__ __attribute__((aligned(16))) uint8_t sm[];    // [2][stage], [2][BT] 2^-e, [BT] 1/rms
    float* esl = (float*)(sm + 2 * kStageBytes);
    float* irms = esl + 2 * BT;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int t0 = blockIdx.x * BT, g0 = blockIdx.x * TT, nt = min(BT, p.n_tok - t0);
    const bool swiglu = p.epi == ORC_EPI_SWIGLU, norm = p.norm_w != nullptr;
    const uint8_t *const sw0 = spin(p.w[0]), *const sw1 = spin(p.w[1]), *const sw2 = spin(p.w[2]);
    const int n_seg = p.n_seg, r0 = p.rows[0], r1 = p.rows[1], n_blk = p.n_in / 32;
    // the lane's logical row (past the end: row 0 is read, nothing written)
    const int rb = blockIdx.y * RW + wave, jo = rb * 16 + (n & 15);
    const int jl = swiglu ? (jo < r0 ? (n >> 4) * r0 + jo : p.n_rows) : rb * 32 + n;
    const uint8_t* rp;
    {
        int jj;
        const int sg = seg_of(jl < p.n_rows ? jl : 0, n_seg, r0, r1, jj);
        rp = pick3(sg, sw0, sw1, sw2) + (size_t)jj * p.row_bytes;
    }

    // stage st's fragments straight into the LDS (its buffer's readers are
    // done); the powers of a superblock with its first stage
    float es_n = 1.f;
    auto a_load = [&](int st) {
        uint8_t* const d = sm + (st & 1) * kStageBytes;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int f = wave + i * RW, g = f / (4 * PL), o = f % (4 * PL);
            const uint8_t* src = wk.frag + ((size_t)(g0 + g) * wk.stages + st) * kGrpStage + o * kFragBytes;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + lane * 16),
                                             (__attribute__((address_space(3))) void*)(d + f * kFragBytes), 16, 0, 0);
        }
        if ((st & 3) == 0 && tid < BT) es_n = *(gfp)(wk.es + ((size_t)(g0 + (tid >> 5)) * wk.supers + (st >> 2)) * 32 + (tid & 31));
    };
    auto es_store = [&](int st) {
        if ((st & 3) == 0 && tid < BT) esl[((st >> 2) & 1) * BT + tid] = es_n;
    };

    f16v acc[TT], D[TT];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[tt][e] = D[tt][e] = 0.f;

    Row cur, nxt;
    const int S0 = 4 * (int)((size_t)wk.supers * blockIdx.z / gridDim.z);
    const int S1 = min(wk.stages, 4 * (int)((size_t)wk.supers * (blockIdx.z + 1) / gridDim.z));
    a_load(S0);
    nxt.load(rp, S0, h, n_blk);
    es_store(S0);

    // one stage: its fragments from the LDS against the row's codes, one
    // (block, token tile) after another; a tile's fragments are asked for ahead
    // of the products of the tile before (the compiler moves the reads down to
    // that tile's last product, which is all that covers them). The scheduling
    // barriers keep it from starting more tiles at once than the registers
    // hold.
    auto stage = [&](int st, int gb) {  // gb: first block of the stage in the granule
        const uint8_t* ab = sm + (st & 1) * kStageBytes + lane * 16;
        h8v av[2][2][PL], bh[2], bl[2];
        float d = 1.f;
        auto read = [&](int i) {
            const int b = i / TT, tt = i % TT;
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int pl = 0; pl < PL; ++pl)
                    av[i & 1][a][pl] = *(const h8v*)(ab + tt * kGrpStage + ((2 * b + a) * PL + pl) * kFragBytes);
        };
        read(0);
#pragma unroll
        for (int i = 0; i < 2 * TT; ++i) {
            if (i % TT == 0) {
                cur.block(gb + i / TT, st, h);
#pragma unroll
                for (int a = 0; a < 2; ++a) cur.step(gb + i / TT, a, bh[a], bl[a]);
                d = i / TT ? -cur.scale() : cur.scale();  // odd blocks are stored negated
            }
            if (i + 1 < 2 * TT) read(i + 1);
            f16v c;
#pragma unroll
            for (int e = 0; e < 16; ++e) c[e] = 0.f;
            if constexpr (Row::SPLIT) {  // hi activations x code remainders (lo x lo is below 2^-22)
#pragma unroll
                for (int a = 0; a < 2; ++a) c = mfma<Row::BF>(av[i & 1][a][0], bl[a], c);
            }
#pragma unroll
            for (int pl = PL - 1; pl >= 0; --pl)
#pragma unroll
                for (int a = 0; a < 2; ++a) c = mfma<Row::BF>(av[i & 1][a][pl], bh[a], c);
#pragma unroll
            for (int e = 0; e < 16; ++e) D[i % TT][e] = __builtin_fmaf(d, c[e], D[i % TT][e]);
            asm volatile("" : "+v"(D[i % TT]));  // joined here (else every tile's c stays live to a later block)
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // end of a superblock: (Q4_K: the sub-block sums' part, then) acc += 2^-e D
    auto flush = [&](int sb) {
        const float* el = esl + (sb & 1) * BT;
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            if constexpr (Row::MINS) {
                h8v sc8, mn8;
                cur.scales(sc8, mn8);
                const uint8_t* sp = wk.sums + ((size_t)(g0 + tt) * wk.supers + sb) * (2 * kFragBytes) + lane * 16;
                const h8v s0 = __builtin_bit_cast(h8v, ldg16(sp)), s1 = __builtin_bit_cast(h8v, ldg16(sp + kFragBytes));
                f16v z, y;
#pragma unroll
                for (int e = 0; e < 16; ++e) z[e] = y[e] = 0.f;
                z = mfma<false>(s1, sc8, z);
                z = mfma<false>(s0, sc8, z);
                y = mfma<false>(s1, mn8, y);
                y = mfma<false>(s0, mn8, y);
                // the sums are stored times 2^-6
                const float d8 = 512.f * cur.scale(), dm = -64.f * cur.dmin();
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    D[tt][e] = __builtin_fmaf(d8, z[e], __builtin_fmaf(dm, y[e], D[tt][e]));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 e4 = *(const float4*)(el + tt * 32 + 8 * i + 4 * h);
                const float es[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int e = 4 * i + k;
                    acc[tt][e] = __builtin_fmaf(es[k], D[tt][e], acc[tt][e]);
                    D[tt][e] = 0.f;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    for (int st = S0; st < S1; st += 2) {  // whole 128-value units
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int s = st + k;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies of stage s
            __syncthreads();  // stage s is in the LDS; the other buffer's readers are done
            if (k % GR == 0) cur = nxt;
            if (s + 1 < S1) a_load(s + 1);
            if (k % GR == 0 && s + GR < S1) nxt.load(rp, s + GR, h, n_blk);
            stage(s, GR == 2 ? 2 * k : 0);
            if (k == 1 && ((s & 3) == 3 || s + 1 == S1)) flush(s >> 2);
            if (s + 1 < S1) es_store(s + 1);
        }
    }

    // lane (n, h) holds tokens 8 (e / 4) + 4 h + e % 4 of each token tile, row jl
    if (part) {
        if (jl < p.n_rows) {
            float* o = part + ((size_t)blockIdx.z * p.n_tok + t0) * p.n_rows + jl;
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int tl = tt * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
                    if (tl < nt) *(gwp)(o + (size_t)tl * p.n_rows) = acc[tt][e];
                }
        }
        return;
    }
    // 1 / rms of each token from its superblocks' sums of x^2
    if (norm) {
        if (tid < BT) irms[tid] = pf_inv_rms(wk, g0 + (tid >> 5), tid & 31, p.n_in, p.eps);
        __syncthreads();
    }
    float *const sy0 = spin(p.y[0]), *const sy1 = spin(p.y[1]), *const sy2 = spin(p.y[2]);
    const float *const sb0 = spin(p.bias[0]), *const sb1 = spin(p.bias[1]), *const sb2 = spin(p.bias[2]);
    int jj;
    const int sg = seg_of(jl < p.n_rows ? jl : 0, n_seg, r0, r1, jj);
    float* y = swiglu ? sy0 + jo : pick3(sg, sy0, sy1, sy2) + jj;
    const float* bb = pick3(sg, sb0, sb1, sb2);
    const float bias = bb && !swiglu ? *(gfp)(bb + jj) : 0.f;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int tl = tt * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
            const float v = acc[tt][e] * (norm ? irms[tl] : 1.f);
            const float u = swiglu ? __shfl_xor(v, 16, 64) : 0.f;  // the gate row's up row
            if (tl >= nt || jl >= p.n_rows || (swiglu && n >= 16)) continue;
            pf_write(p, y + (size_t)(t0 + tl) * p.ldy, v, u, bb ? bias : 0.f);
        }
}

// Sum of the ranges' partial results in range order, then the epilogue: four
// output values per thread, the loads of four ranges in flight. Bound by
// memory (a few MB).
constexpr int kSumV = 4;
__global__ __launch_bounds__(256) void k_pf_sum(QmvParams p, PfWork wk, const float* part, int nz) {
    const int tok = blockIdx.y, j0 = blockIdx.x * (256 * kSumV) + threadIdx.x;
    const bool swiglu = p.epi == ORC_EPI_SWIGLU;
    const int rows = swiglu ? p.rows[0] : p.n_rows;
    const size_t zs = (size_t)p.n_tok * p.n_rows;
    auto sum = [&](const float* s, float (&v)[kSumV]) {
#pragma unroll
        for (int k = 0; k < kSumV; ++k) v[k] = 0.f;
        for (int z0 = 0; z0 < nz; z0 += 4) {
            float t[4][kSumV];
#pragma unroll
            for (int z = 0; z < 4; ++z)
#pragma unroll
                for (int k = 0; k < kSumV; ++k)
                    t[z][k] = *(gfp)(s + min(z0 + z, nz - 1) * zs + min(j0 + 256 * k, rows - 1));
#pragma unroll
            for (int z = 0; z < 4; ++z)
#pragma unroll
                for (int k = 0; k < kSumV; ++k)
                    if (z0 + z < nz) v[k] += t[z][k];
        }
    };
    float v[kSumV], u[kSumV];
    const float* s = part + (size_t)tok * p.n_rows;
    sum(s, v);
    if (swiglu) sum(s + rows, u);
    const float inv = p.norm_w ? pf_inv_rms(wk, tok >> 5, tok & 31, p.n_in, p.eps) : 1.f;
#pragma unroll
    for (int k = 0; k < kSumV; ++k) {
        const int j = j0 + 256 * k;
        if (j >= rows) continue;
        int jj;
        const int sg = seg_of(j, p.n_seg, p.rows[0], p.rows[1], jj);
        float* y = swiglu ? p.y[0] + j : pick3(sg, p.y[0], p.y[1], p.y[2]) + jj;
        const float* bb = swiglu ? nullptr : pick3(sg, p.bias[0], p.bias[1], p.bias[2]);
        pf_write(p, y + (size_t)tok * p.ldy, v[k] * inv, swiglu ? u[k] * inv : 0.f, bb ? bb[jj] : 0.f);
    }
}

// ── workspace ────────────────────────────────────────────────────────────────
// One per device, allocated by orc_init and freed by orc_shutdown (or when
// orc_init selects another device). A call holds the lock while it enqueues
// its launches, and its stream first waits for the last use on any other
// stream, so calls of any streams and threads take the workspace in turn.
// Uses that follow each other on one of the library's own streams need no
// event: it is recorded when another stream wants the workspace (which then
// also waits for what the first stream has enqueued since), when a capture of
// the stream begins (orc_graph_begin, under the lock: the event must not
// become part of the capture) or when the stream is destroyed. An event after
// every use costs 4.4 us of GPU time between two calls (3B blocks at 127
// tokens: 22 of 222 us a layer). A stream the library did not create may be
// destroyed behind its back, so its uses are followed by an event at once.
// GEMM calls that need more than kPfWorkBytes go in token chunks. A device
// without that much memory left has no workspace: calls take the kernels that
// do without.
static std::mutex g_pf_mu;
static uint8_t* g_pf_buf = nullptr;
static hipEvent_t g_pf_ev = nullptr;
static bool g_pf_ev_set = false;         // g_pf_ev follows the last use
static hipStream_t g_pf_last = nullptr;  // or the last use is on this stream of the library

static hipError_t pf_new_event(hipEvent_t* ev) {
    return hipEventCreateWithFlags(ev, hipEventDisableTiming | hipEventDisableSystemFence);
}

void pf_release() {
    std::lock_guard<std::mutex> lk(g_pf_mu);
    if (g_pf_buf) (void)hipFree(g_pf_buf);
    if (g_pf_ev) (void)hipEventDestroy(g_pf_ev);
    g_pf_buf = nullptr;
    g_pf_ev = nullptr;
    g_pf_ev_set = false;
    g_pf_last = nullptr;
}

int pf_init() {
    pf_release();
    std::lock_guard<std::mutex> lk(g_pf_mu);
    ORC_HIP_CHECK(pf_new_event(&g_pf_ev));
    if (hipMalloc((void**)&g_pf_buf, kPfWorkBytes) != hipSuccess) {
        g_pf_buf = nullptr;
        (void)hipGetLastError();  // not the next launch's error
    }
    return ORC_OK;
}

static bool capturing(hipStream_t s) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone;
}

int pf_ws_begin(hipStream_t s, uint8_t** buf) {
    std::unique_lock<std::mutex> lk(g_pf_mu);
    if (!g_pf_buf || capturing(s)) return kPfBusy;
    if (g_pf_last != s) {
        if (g_pf_last) {
            // A capture of that stream that was begun through HIP itself: no
            // event of it can be waited for, and it may begin between the
            // question and the record. The event is then part of the capture:
            // another one takes its place.
            if (capturing(g_pf_last)) return kPfBusy;
            ORC_HIP_CHECK(hipEventRecord(g_pf_ev, g_pf_last));
            if (capturing(g_pf_last)) {
                hipEvent_t ev;
                ORC_HIP_CHECK(pf_new_event(&ev));
                (void)hipEventDestroy(g_pf_ev);
                g_pf_ev = ev;
                return kPfBusy;
            }
            g_pf_last = nullptr;
            g_pf_ev_set = true;
        }
        if (g_pf_ev_set) ORC_HIP_CHECK(hipStreamWaitEvent(s, g_pf_ev, 0));
    }
    *buf = g_pf_buf;
    lk.release();  // held until pf_ws_end
    return ORC_OK;
}

int pf_ws_end(hipStream_t s) {
    std::unique_lock<std::mutex> lk(g_pf_mu, std::adopt_lock);
    if (library_stream(s)) {
        g_pf_last = s;
        return ORC_OK;
    }
    g_pf_last = nullptr;
    g_pf_ev_set = true;
    ORC_HIP_CHECK(hipEventRecord(g_pf_ev, s));
    return ORC_OK;
}

int pf_ws_capture(hipStream_t s) {
    std::lock_guard<std::mutex> lk(g_pf_mu);
    if (g_pf_last == s && !capturing(s)) {
        ORC_HIP_CHECK(hipEventRecord(g_pf_ev, s));
        g_pf_last = nullptr;
        g_pf_ev_set = true;
    }
    ORC_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    return ORC_OK;
}

void pf_ws_forget(hipStream_t s) {
    std::lock_guard<std::mutex> lk(g_pf_mu);
    if (g_pf_last != s) return;
    g_pf_last = nullptr;
    g_pf_ev_set = hipEventRecord(g_pf_ev, s) == hipSuccess;
}

struct PfType {
    int pieces;
    bool perm, sums;
};
static bool pf_type(int type, PfType& t) {
    switch (type) {
        case ORC_Q4_K: t = {2, true, true}; return true;
        case ORC_Q6_K:
        case ORC_Q8_0:
        case ORC_Q8_0_X8:
        case ORC_Q4_0: t = {2, true, false}; return true;
        case ORC_F16: t = {2, false, false}; return true;
        case ORC_BF16: t = {3, false, false}; return true;
        default: return false;
    }
}

// Workspace bytes of ng token groups, and the arrays inside buf.
static size_t pf_layout(const PfType& t, int n_in, int ng, uint8_t* buf, PfWork& w) {
    w.stages = (n_in + 127) / 128 * 2;
    w.supers = (n_in + kSuper - 1) / kSuper;
    const size_t frag = (size_t)ng * w.stages * 4 * t.pieces * kFragBytes, side = (size_t)ng * w.supers * 32 * sizeof(float);
    const size_t sums = t.sums ? (size_t)ng * w.supers * 2 * kFragBytes : 0;
    w.frag = buf;
    w.sums = buf + frag;
    w.es = (float*)(buf + frag + sums);
    w.ss = (float*)(buf + frag + sums + side);
    return frag + sums + 2 * side;
}

template <int QT, int RW, int TT>
static int pf_shape(const QmvParams& p, const PfWork& w, int nz, float* part, hipStream_t s, hipEvent_t stop) {
    constexpr int BT = 32 * TT;
    const bool swiglu = p.epi == ORC_EPI_SWIGLU;
    const int rows_blk = (swiglu ? 16 : 32) * RW, rows = swiglu ? p.rows[0] : p.n_rows;
    const dim3 grid((p.n_tok + BT - 1) / BT, (rows + rows_blk - 1) / rows_blk, nz);
    const size_t lds = 2 * (size_t)TT * 4 * PfRow<QT>::PL * kFragBytes + 3 * BT * sizeof(float);
    float* const pt = nz > 1 ? part : nullptr;
    const hipEvent_t st = pt ? nullptr : stop;
    if (grid.y > 65535) return set_error(ORC_E_UNSUPPORTED, "gemm: too many rows for a prefill launch");
    if (st)
        hipExtLaunchKernelGGL((k_pf<QT, RW, TT>), grid, dim3(64 * RW), lds, s, nullptr, st, 0, p, w, pt);
    else
        hipLaunchKernelGGL((k_pf<QT, RW, TT>), grid, dim3(64 * RW), lds, s, p, w, pt);
    ORC_LAUNCH_CHECK();
    if (!pt) return ORC_OK;
    const dim3 g2((rows + 256 * kSumV - 1) / (256 * kSumV), p.n_tok);
    if (stop) hipExtLaunchKernelGGL(k_pf_sum, g2, dim3(256), 0, s, nullptr, stop, 0, p, w, (const float*)part, nz);
    else hipLaunchKernelGGL(k_pf_sum, g2, dim3(256), 0, s, p, w, (const float*)part, nz);
    ORC_LAUNCH_CHECK();
    return ORC_OK;
}

// Tile shape and number of K ranges of a launch, from sweeps of the 0.5B, 1B,
// 3B and 7B layer matrices at 20 to 1023 tokens (us, MI355X; rows x n_in,
// type, tokens):
//  * 128 rows x 32 tokens for at most 32 tokens (7B gate+up Q6_K 75 against
//    90 with 64-token tiles), and for narrow matrices, where 64-token tiles in
//    the most ranges below leave CUs idle: such a launch is one wave per SIMD
//    and as long as its chain of dependent products, which a 32-token tile
//    halves (896 x 896 Q8_0 in four ranges: 14.0 at 64 tokens, 16.0 at 256
//    and 19.4 at 512 against 20.4, 28.6 and 28.9 with 64-token tiles; 1023
//    tokens, one range, 24.9 against 30.4; 896 x 4864 at 256 27.5 against
//    30.0; 3072 x 3072 Q4_K at 48 19.7 against 20.9);
//  * 128 x 128 once such tiles are two per CU (7B gate+up, 1023 tokens: 891
//    against 1024 with 128 x 64; 2048-wide Q4_0 216 against 270) and K is at
//    least eight superblocks (0.5B gate+up, n_in 896: 110 against 87), not
//    for BF16, whose three pieces per value leave one such workgroup per CU
//    (332 against 262);
//  * 128 x 64 otherwise (3072 x 3072 Q4_K, 1023 tokens: 84 against 107).
//  * K is split while the tiles leave CUs idle: up to 768 workgroups (three
//    per CU, which the 64-token kernels of Q4_K, Q8_0, Q4_0 and F16 allow; Q6_K
//    and BF16 hold 177 and 172 registers, two per CU), ranges of at least two
//    superblocks (three above 128 tokens, where the partial
//    sums weigh more); with 32-token tiles up to 512 workgroups, and a short
//    K in up to four ranges (896 x 896 at 256 tokens: 22.6, 18.6, 17.6 and
//    16.1 in one to four). 3584 x 18944 at 127 tokens 364 in one range, 106 in
//    eight; 3584 x 3584 83 -> 38; F16 2048 x 8192 142 -> 34. F16 and BF16
//    rows are cut at 16 superblocks at any size: the rounding of one long
//    chain would exceed the fp32 kernel's (8192 values: 1.35e-7 of the
//    result in one range, 1.1e-7 in two, 1.33e-7 there).
constexpr int kDenseSupers = 16;
static bool pf_dense(int type) { return type == ORC_F16 || type == ORC_BF16; }
struct PfPlan {
    int shape, nz;  // shape 0: 128 x 128, 1: 128 x 64, 2: 128 x 32
};
static PfPlan pf_plan(int type, const QmvParams& p, int supers) {
    const int rows = p.epi == ORC_EPI_SWIGLU ? 2 * p.rows[0] : p.n_rows;
    auto wgs = [&](int bt) { return (long)((rows + 127) / 128) * ((p.n_tok + bt - 1) / bt); };
    PfPlan r{1, 1};
    const int most = std::min(16, std::max(1, (supers + 1) / (p.n_tok <= 128 ? 2 : 3)));
    if (p.n_tok <= 32 || wgs(64) * most < g_n_cu) r.shape = 2;
    else if (type != ORC_BF16 && p.n_tok > 64 && supers >= 8 && wgs(128) >= 2 * g_n_cu) r.shape = 0;
    if (r.shape == 2)
        r.nz = (int)std::min<long>(std::max(most, std::min(supers, 4)), 2 * g_n_cu / wgs(32));
    else
        r.nz = (int)std::min<long>(most, 3 * g_n_cu / wgs(r.shape == 0 ? 128 : 64));
    r.nz = std::max(r.nz, 1);
    if (pf_dense(type)) r.nz = std::max(r.nz, (supers + kDenseSupers - 1) / kDenseSupers);
    return r;
}

// Microseconds of a launch pair by its longest chain: per superblock of a range
// 2.7 (4.8 for rows whose loads wait for each other), 3 more with 64-token
// tiles, per round of workgroups 3.5, the sum of the ranges 1.6 + 0.15 each; the
// norm 1, SwiGLU 1.5, the launches of a second weight type 6.
// Within 5% (rms) of the measured times of 61 matrices of 64 to 8192 rows and
// 256 to 8192 values at 24 to 255 tokens, up to about 25 us; above that the
// products count, and it is far too low.
double pf_estimate(int type, const QmvParams& p) {
    const int supers = (p.n_in + kSuper - 1) / kSuper;
    double us = 3.5 + (p.norm_w ? 1.0 : 0.0) + (p.epi == ORC_EPI_SWIGLU ? 1.5 : 0.0);
    for (int i0 = 0; i0 < p.n_seg;) {
        QmvParams q = p;
        int i1 = i0;
        q.n_rows = 0;
        for (; i1 < p.n_seg && p.seg_type[i1] == p.seg_type[i0]; ++i1) q.n_rows += p.rows[i1];
        const int ty = p.seg_type[i0];
        const PfPlan r = pf_plan(ty, q, supers);
        const int bt = r.shape == 0 ? 128 : r.shape == 1 ? 64 : 32;
        const int rows = p.epi == ORC_EPI_SWIGLU ? 2 * p.rows[0] : q.n_rows;
        const long wgs = (long)((rows + 127) / 128) * ((p.n_tok + bt - 1) / bt) * r.nz;
        const bool serial = ty == ORC_Q8_0 || ty == ORC_Q8_0_X8 || ty == ORC_Q4_0;
        us += (i0 ? 6.0 : 0.0) + 3.5 * ((wgs + g_n_cu - 1) / g_n_cu) + ((serial ? 4.8 : 2.7) + (r.shape == 2 ? 0 : 3)) * ((supers + r.nz - 1) / r.nz);
        if (r.nz > 1) us += 1.6 + 0.15 * r.nz;
        i0 = i1;
    }
    return us;
}

template <int QT>
static int pf_run(const QmvParams& p, const PfWork& w, const PfPlan& r, float* part, hipStream_t s, hipEvent_t stop) {
    if constexpr (QT != ORC_BF16)
        if (r.shape == 0) return pf_shape<QT, 4, 4>(p, w, r.nz, part, s, stop);
    return r.shape == 1 ? pf_shape<QT, 4, 2>(p, w, r.nz, part, s, stop) : pf_shape<QT, 4, 1>(p, w, r.nz, part, s, stop);
}

static int pf_split(const PfType& t, const PfSplit& sp, int ng, hipStream_t s, hipEvent_t start) {
    const dim3 grid(sp.w.supers, ng);
    auto go = [&](auto kern) {
        if (start) hipExtLaunchKernelGGL(kern, grid, dim3(256), 0, s, start, nullptr, 0, sp);
        else hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, sp);
    };
    if (t.pieces == 3) go(k_pf_split<3, false, false>);
    else if (t.sums) go(k_pf_split<2, true, true>);
    else if (t.perm) go(k_pf_split<2, true, false>);
    else go(k_pf_split<2, false, false>);
    ORC_LAUNCH_CHECK();
    return ORC_OK;
}

// Tokens of a chunk: as many as fit the workspace, with the partial sums of the
// ranges that a long F16 or BF16 row needs (a chunk of fewer tokens otherwise,
// down to 64; 0: not even those). Other partial sums take what is left.
static int pf_chunk(int type, const PfType& t, const QmvParams& p) {
    PfWork w;
    const int supers = (p.n_in + kSuper - 1) / kSuper, nz = pf_dense(type) ? (supers + kDenseSupers - 1) / kDenseSupers : 1;
    const size_t tok = nz > 1 ? (size_t)nz * p.n_rows * sizeof(float) : 0;
    const size_t per = pf_layout(t, p.n_in, 4, nullptr, w) + 128 * tok;
    if (per <= kPfWorkBytes) return (int)std::min<size_t>(kPfWorkBytes / per, 1 << 20) * 128;
    return pf_layout(t, p.n_in, 2, nullptr, w) + 64 * tok <= kPfWorkBytes ? 64 : 0;
}

constexpr int kPfMaxRows = 65535 * 128;

bool pf_takes(int type, const QmvParams& p) {
    if (p.n_tok < kPfSplitMin || p.n_in % 32) return false;
    PfType t;
    if (type == kMixK) t = {2, true, true};
    else if (!pf_type(type, t)) return false;
    if (p.epi == ORC_EPI_SWIGLU && p.n_seg != 2) return false;
    // blocks of 128 rows (64 SwiGLU pairs) are the second grid dimension
    if (p.n_rows > kPfMaxRows) return false;
    return pf_chunk(type, t, p) > 0;
}

int pf_launch(int type, const QmvParams& p0, hipStream_t s, const LaunchEvents& ev, uint8_t* buf) {
    PfType t;
    if (type == kMixK) t = {2, true, true};  // Q4_K and Q6_K segments share one split
    else if (!pf_type(type, t)) return set_error(ORC_E_INVALID, "gemm: not a prefill launch");
    PfWork w;
    const int chunk = pf_chunk(type, t, p0);
    int rc = ORC_OK;
    for (int t0 = 0; t0 < p0.n_tok && !rc; t0 += chunk) {
        QmvParams p = p0;
        p.n_tok = std::min(chunk, p0.n_tok - t0);
        p.x = p0.x + (size_t)t0 * p0.ldx;
        for (int i = 0; i < 3; ++i) p.y[i] = p0.y[i] ? p0.y[i] + (size_t)t0 * p0.ldy : nullptr;
        const int ng = p.n_tok <= 64 ? 2 : (p.n_tok + 127) / 128 * 4;
        const size_t used = pf_layout(t, p.n_in, ng, buf, w);
        PfSplit sp{w, p.x, p.norm_w, p.ldx, p.n_tok, p.n_in};
        if ((rc = pf_split(t, sp, ng, s, t0 == 0 ? ev.start : nullptr))) break;
        // one launch per run of segments of one type
        for (int i0 = 0; i0 < p.n_seg && !rc;) {
            int i1 = i0 + 1;
            while (i1 < p.n_seg && p.seg_type[i1] == p.seg_type[i0]) ++i1;
            QmvParams q = p;
            q.n_seg = i1 - i0;
            q.n_rows = 0;
            for (int i = 0; i < 3; ++i) {
                const bool in = i < q.n_seg;
                q.w[i] = in ? p.w[i0 + i] : nullptr;
                q.y[i] = in ? p.y[i0 + i] : nullptr;
                q.bias[i] = in ? p.bias[i0 + i] : nullptr;
                q.rows[i] = in ? p.rows[i0 + i] : 0;
                q.n_rows += q.rows[i];
            }
            q.row_bytes = p.seg_rb[i0];
            const hipEvent_t stop = i1 == p.n_seg && t0 + chunk >= p0.n_tok ? ev.stop : nullptr;
            PfPlan r = pf_plan(p.seg_type[i0], q, w.supers);
            float* const part = (float*)(buf + used);  // partial sums behind the split activations
            r.nz = (int)std::min<size_t>(r.nz, std::max<size_t>(1, (kPfWorkBytes - used) / ((size_t)p.n_tok * q.n_rows * 4)));
            switch (p.seg_type[i0]) {
                case ORC_Q4_K: rc = pf_run<ORC_Q4_K>(q, w, r, part, s, stop); break;
                case ORC_Q6_K: rc = pf_run<ORC_Q6_K>(q, w, r, part, s, stop); break;
                case ORC_Q8_0: rc = pf_run<ORC_Q8_0>(q, w, r, part, s, stop); break;
                case ORC_Q8_0_X8: rc = pf_run<ORC_Q8_0_X8>(q, w, r, part, s, stop); break;
                case ORC_Q4_0: rc = pf_run<ORC_Q4_0>(q, w, r, part, s, stop); break;
                case ORC_F16: rc = pf_run<ORC_F16>(q, w, r, part, s, stop); break;
                case ORC_BF16: rc = pf_run<ORC_BF16>(q, w, r, part, s, stop); break;
                default: rc = set_error(ORC_E_UNSUPPORTED, "gemm: not a prefill type");
            }
            i0 = i1;
        }
    }
    return rc;
}

}  // namespace orc
