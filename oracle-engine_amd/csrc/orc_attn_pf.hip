// Prefill attention on the fp16 matrix cores (gfx950): RoPE, K / V store and
// causal GQA attention of a prompt pass (core/model.cpp:595-626) for
// orc_attn_prefill, in two or three launches over the library's workspace:
//  * k_kv_split stores the pass's K (rotated) and V rows in the cache and
//    writes every cached position's K and V once more as MFMA fragments: each
//    value a power of two per 32 positions times (hi = fp16, lo = fp16 of the
//    rest), ~22 bits.
//  * k_attn_fa: a workgroup takes 32 RT rows (token, query head) of one kv
//    head through the key blocks with an online softmax. Scores are formed
//    transposed (keys x rows), so a lane holds one row's scores and the
//    probabilities are already the next product's operand: nothing crosses
//    lanes but one maximum per block.
//  * k_attn_fa_sum merges key ranges where few rows leave CUs idle.
// Products: hi x hi + hi x lo + lo x hi of exact fp16 halves, 3/16 of the time
// of the fp32 MFMA chains of k_attn_pf (which stays for captured calls, for
// caches larger than the workspace and for short contexts, attn_short). Every
// factor keeps ~22 bits against fp32's 24; the error against 64 bits is lower
// all the same, since the sums are better (7B shape, 1023 tokens at 3000:
// 2.8e-7 of the result against 1.14e-6; 3B, 127 at 0: 1.5e-7 against 2.7e-7).
// Sums: the matrix cores round toward minus infinity, so every block's
// products start from zero (the small ones apart for the scores, first for
// P V), the blocks are added up in fp32 on the vector ALUs, and K and V are
// stored negated in two of every four blocks.
// Range: a block's probabilities are formed against its own row maximum
// (rounded up to a whole power of two from the first block's) and V against its
// own, so both halves of a product hold their bits whatever the other blocks
// weigh; the running O and sum keep their powers of two as integers, so adding
// a block up rounds nothing but the sums themselves. Inside a block one power of two serves all
// 32 positions: a block where some K or V row's largest value is below 2^-16
// of the block's (its halves would keep fewer than 22 bits), or that holds an
// infinity or NaN (which must not reach rows that do not see the position: 0
// times infinity), is marked, and the waves take it in fp32 from the cache.
#include "orc_gemm.hpp"
#include "orc_attn_pf.hpp"

#include <algorithm>

namespace orc {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(1))) float* gfp;

constexpr int kKB = 32;  // key positions per block
constexpr int kPlain = 1024;  // an exponent's range is -128 .. 127
template <int HD> constexpr int fa_block_bytes() { return HD * 256; }  // K and V fragments of a block

// rotate-half of the pair (a, b) by (cos, sin): the rounding of every row rotation
__device__ __forceinline__ float rot_lo(float a, float b, float2 cs) { return __builtin_fmaf(a, cs.x, -(b * cs.y)); }
__device__ __forceinline__ float rot_hi(float a, float b, float2 cs) { return __builtin_fmaf(b, cs.x, a * cs.y); }

__device__ __forceinline__ int sign_of(int blk) { return (blk >> 1) & 1; }  // 1: stored negated

// exponent e with |v| 2^e below 2^14 for |v| <= mx
__device__ __forceinline__ int up_exp(float mx) {
    if (!(mx > 0.f)) return 0;
    int ex;
    (void)frexpf(mx, &ex);
    return max(-120, min(14 - ex, 120));
}

__device__ __forceinline__ uint32_t split2(float a, float b, uint32_t& lo) {
    const h2v hi = __builtin_convertvector((f2v){a, b}, h2v);
    f2v r = {a - (float)hi.x, b - (float)hi.y};
    if (!(fabsf(a) <= 3.4028234e38f)) r.x = 0.f;  // an infinity or NaN is its hi half alone
    if (!(fabsf(b) <= 3.4028234e38f)) r.y = 0.f;
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, h2v));
    return __builtin_bit_cast(uint32_t, hi);
}

struct FaWork {
    uint8_t* frag;  // [kv head][block] fragments: K [dims 16 s][hi, lo], V [dims 32 dt][keys 16 s][hi, lo], 1 KB each
    int* exps;      // [kv head][block]: exponents of the stored K (times 2^16) and V (value = stored 2^-exp), plus
                    // kPlain where the block is taken in fp32
    int n_blk;
};

// Grid (block, kv head), 2 HD threads. K: thread = (key, 16 dims); V: thread =
// (dim, 16 keys). A V fragment's K order is the one the scores come in: half h,
// slot j = key 16 s + 8 (j / 4) + 4 h + j % 4. Bound by memory (each row read
// and written once).
template <int HD>
__global__ __launch_bounds__(2 * HD) void k_kv_split(const float* qkv, int ldqkv, int n_heads, int n_kv, int start,
                                                     int p_end, const float2* rope, float* kc, float* vc, int ctx,
                                                     FaWork w) {
    constexpr int half = HD / 2, HS = HD / 32;
    __shared__ float red[2][2 * HD / 64];
    __shared__ uint32_t rows[2 * HD / 64][5];
    const int blk = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
    const size_t kcol = (size_t)(n_heads + g) * HD, vcol = (size_t)(n_heads + n_kv + g) * HD;
    // every load first, without branches between them (positions past the end
    // read the last one): one round trip instead of one per position
    const int key = tid & 31, s = tid >> 5, p = blk * kKB + key, pc = min(p, p_end - 1), sl = s & (HS - 1);
    const bool mine = p >= start;  // a row of this pass: rotated, stored in the cache
    const float* kra = mine ? qkv + (size_t)(pc - start) * ldqkv + kcol + 16 * sl : kc + ((size_t)g * ctx + pc) * HD + 16 * s;
    const float* krb = mine ? kra + half : kra;
    const float4* cs = (const float4*)(rope + (size_t)pc * half + 16 * sl);
    float4 ka[4], kb[4], c[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) ka[i] = ((const float4*)kra)[i], kb[i] = ((const float4*)krb)[i];
#pragma unroll
    for (int i = 0; i < 8; ++i) c[i] = cs[i];
    const int d = tid % HD, s2 = tid / HD;
    float vv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int pv = min(blk * kKB + 16 * s2 + i, p_end - 1);
        vv[i] = *(pv < start ? vc + ((size_t)g * ctx + pv) * HD + d : qkv + (size_t)(pv - start) * ldqkv + vcol + d);
    }
    float kv[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float av[4] = {ka[i].x, ka[i].y, ka[i].z, ka[i].w}, bv[4] = {kb[i].x, kb[i].y, kb[i].z, kb[i].w};
        const float2 cv[4] = {{c[2 * i].x, c[2 * i].y}, {c[2 * i].z, c[2 * i].w}, {c[2 * i + 1].x, c[2 * i + 1].y}, {c[2 * i + 1].z, c[2 * i + 1].w}};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float r = s < HS ? rot_lo(av[k], bv[k], cv[k]) : rot_hi(av[k], bv[k], cv[k]);
            kv[4 * i + k] = p < p_end ? (mine ? r : av[k]) : 0.f;
        }
    }
    if (mine && p < p_end) {
        float4* dst = (float4*)(kc + ((size_t)g * ctx + p) * HD + 16 * s);
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[i] = make_float4(kv[4 * i], kv[4 * i + 1], kv[4 * i + 2], kv[4 * i + 3]);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int pv = blk * kKB + 16 * s2 + i;
        if (pv >= start && pv < p_end) vc[((size_t)g * ctx + pv) * HD + d] = vv[i];
        if (pv >= p_end) vv[i] = 0.f;
    }
    float mk = 0.f, mv = 0.f, rk;
    bool odd = false;
#pragma unroll
    for (int i = 0; i < 16; ++i) {  // infinities and NaN set no scale
        const float a = fabsf(kv[i]), b = fabsf(vv[i]);
        odd |= !(a <= 3.4028234e38f) || !(b <= 3.4028234e38f);
        mk = fmaxf(mk, a <= 3.4028234e38f ? a : 0.f);
        mv = fmaxf(mv, b <= 3.4028234e38f ? b : 0.f);
    }
    rk = mk;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        mk = fmaxf(mk, __shfl_xor(mk, o, 64));
        mv = fmaxf(mv, __shfl_xor(mv, o, 64));
    }
    if ((tid & 63) == 0) red[0][tid >> 6] = mk, red[1][tid >> 6] = mv;
    __syncthreads();
    mk = red[0][0], mv = red[1][0];
#pragma unroll
    for (int i = 1; i < 2 * HD / 64; ++i) mk = fmaxf(mk, red[0][i]), mv = fmaxf(mv, red[1][i]);
    // positions with a value that is not zero, and with one of at least 2^-16
    // of the largest, as bits: K's two rows of lanes hold the same positions,
    // V's lanes hold 16 positions each
    {
        const unsigned long long n2 = __ballot(rk > 0.f), g2 = __ballot(rk >= mk * 0x1p-16f && rk > 0.f);
        uint32_t nv = 0, gv = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float a = fabsf(vv[i]);
            nv |= __ballot(a > 0.f) ? 1u << i : 0u;
            gv |= __ballot(a >= mv * 0x1p-16f && a > 0.f) ? 1u << i : 0u;
        }
        const bool any_odd = __ballot(odd) != 0;
        if ((tid & 63) == 0) {
            uint32_t* d = rows[tid >> 6];
            d[0] = (uint32_t)n2 | (uint32_t)(n2 >> 32), d[1] = (uint32_t)g2 | (uint32_t)(g2 >> 32);
            d[2] = nv << (16 * s2), d[3] = gv << (16 * s2), d[4] = any_odd;
        }
    }
    const int ek = up_exp(mk), ev = mv > 0.f ? up_exp(mv) : 120;  // a block of zeros never sets P V's scale
    const float sg = sign_of(blk) ? -1.f : 1.f, uk = ldexpf(sg, ek), uv = ldexpf(sg, ev);
    uint8_t* f = w.frag + ((size_t)g * w.n_blk + blk) * fa_block_bytes<HD>();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        u32x4 hi, lo;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t l;
            hi[q] = split2(kv[8 * h + 2 * q] * uk, kv[8 * h + 2 * q + 1] * uk, l);
            lo[q] = l;
        }
        uint8_t* o = f + (2 * s) * 1024 + (h * 32 + key) * 16;
        *(u32x4*)o = hi;
        *(u32x4*)(o + 1024) = lo;
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // slots 2q, 2q + 1
            const int k0 = 8 * (q >> 1) + 4 * h + 2 * (q & 1);
            uint32_t l;
            hi[q] = split2(vv[k0] * uv, vv[k0 + 1] * uv, l);
            lo[q] = l;
        }
        o = f + (HD / 16) * 2048 + (((d >> 5) * 2 + s2) * 2) * 1024 + (h * 32 + (d & 31)) * 16;
        *(u32x4*)o = hi;
        *(u32x4*)(o + 1024) = lo;
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t d[5] = {0, 0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 2 * HD / 64; ++i)
#pragma unroll
            for (int k = 0; k < 5; ++k) d[k] |= rows[i][k];
        w.exps[g * w.n_blk + blk] = ek * 65536 + ev + (d[0] != d[1] || d[2] != d[3] || d[4] ? kPlain : 0);
    }
}

// RT row tiles of 32 x KG key groups: wave (rt, kg) takes its 32 rows through
// every KG-th block; the groups are merged in the LDS at the end. Per block
// and wave 3 HD / 16 MFMAs for the scores (32 keys x 32 rows), ~12 vector
// operations per score, 3 HD / 16 MFMAs for P V and HD / 2 vector operations
// to add it up. The blocks (HD / 4 KB each) are copied straight into the LDS,
// the next KG while these multiply.
template <int HD, int RT, int KG>
__global__ __launch_bounds__(64 * RT * KG) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_fa(
    const float* qkv, int ldqkv, int n_tok, int n_heads, int n_kv, int start, const float2* rope, const float* kc,
    const float* vc, int ctx, FaWork w, float* out, int ldo, float* part, int nz) {
    constexpr int half = HD / 2, KS = HD / 16, DT = HD / 32, NW = RT * KG, BB = fa_block_bytes<HD>(), NF = KG * BB / 1024 / NW;
    static_assert(KG * BB / 1024 % NW == 0, "whole fragments");
    extern __shared__ __attribute__((aligned(16))) uint8_t sm[];  // [2][KG][block]
    const int R = n_heads / n_kv, TB = 32 * RT / R;
    const int nb = (n_tok + TB - 1) / TB;
    // kv heads fastest: the workgroups of one kv head land on the same XCDs
    // and share its blocks in their L2; later (longer) token blocks first
    const int g = blockIdx.x % n_kv, tb = nb - 1 - blockIdx.x / n_kv, z = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rt = wave % RT, kg = wave / RT, n = lane & 31, h = lane >> 5;
    const int t0 = tb * TB, nt = min(TB, n_tok - t0), NR = nt * R;
    const int all = (start + t0 + nt + kKB - 1) / kKB;                                         // blocks these rows read
    const int per = (all + nz * KG - 1) / (nz * KG) * KG, b0 = min(all, z * per), b1 = min(all, b0 + per);  // this range's
    const int r = rt * 32 + n, rc = r < NR ? r : 0, ti = rc / R, hd = rc - ti * R, pt = start + t0 + ti;
    const uint8_t* fr = w.frag + (size_t)g * w.n_blk * BB;
    const int* ex = w.exps + g * w.n_blk;

    // copies unrolled in full spill at 128 (39 and 7 registers with one and two
    // row tiles: 127 tokens 22.9 -> 19.3 us without); at 64 they are a little
    // faster (200 tokens at 2000 41.5 -> 40.0)
    constexpr int kUn = HD == 64 ? 16 : 8;
    auto copy = [&](int blk, int buf) {  // blocks blk .. blk + KG - 1 (those below b1)
#pragma unroll kUn
        for (int i = 0; i < NF; ++i) {
            const int f = wave + i * NW, j = f / (BB / 1024);
            if (blk + j < b1)
                __builtin_amdgcn_global_load_lds(
                    (const __attribute__((address_space(1))) void*)(fr + (size_t)blk * BB + f * 1024 + lane * 16),
                    (__attribute__((address_space(3))) void*)(sm + (buf * KG * BB + f * 1024)), 16, 0, 0);
        }
    };
    // this wave's exponents a round ahead, in front of the copies: a wait for
    // them is then no wait for the copies that follow
    int xn = b0 < b1 ? ex[min(b0 + kg, b1 - 1)] : 0;
    if (b0 < b1) copy(b0, 0);

    // the row's rotated query as B operands: dims 16 s + 8 h + 0 .. 7
    h8v qh[KS], ql[KS];
    float cq;  // softmax scale, log2 e and the query's power of two
    {
        const float* q = qkv + (size_t)(t0 + ti) * ldqkv + (size_t)(g * R + hd) * HD + 8 * h;
        const float2* cs = rope + (size_t)pt * half + 8 * h;
        float v[KS][8], mx = 0.f;
#pragma unroll
        for (int s = 0; s < KS / 2; ++s)
#pragma unroll
            for (int j = 0; j < 8; j += 4) {
                const float4 a = *(const float4*)(q + 16 * s + j), b = *(const float4*)(q + half + 16 * s + j);
                const float4 c01 = *(const float4*)(cs + 16 * s + j), c23 = *(const float4*)(cs + 16 * s + j + 2);
                const float av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
                const float2 c[4] = {{c01.x, c01.y}, {c01.z, c01.w}, {c23.x, c23.y}, {c23.z, c23.w}};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    v[s][j + k] = rot_lo(av[k], bv[k], c[k]);
                    v[s + KS / 2][j + k] = rot_hi(av[k], bv[k], c[k]);
                }
            }
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float a = fabsf(v[s][j]);
                mx = fmaxf(mx, a <= 3.4028234e38f ? a : 0.f);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const int eq = up_exp(mx);
        const float uq = ldexpf(1.f, eq);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            u32x4 hi, lo;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t l;
                hi[k] = split2(v[s][2 * k] * uq, v[s][2 * k + 1] * uq, l);
                lo[k] = l;
            }
            qh[s] = __builtin_bit_cast(h8v, hi);
            ql[s] = __builtin_bit_cast(h8v, lo);
        }
        cq = ldexpf(1.4426950408889634f / sqrtf((float)HD), -eq);
    }

    // O^T: dims 32 dt + 8 (e / 4) + 4 h + e % 4 of the lane's row, times 2^(14 - u) and the sign of `last`
    f16v o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
    // m0: the maximum of the row's first block (log2 units). Alone it stays as
    // it is: the largest weight of a row of few keys is 1 exactly. With more
    // blocks to come it is rounded up to a multiple of 2^-16, to which whole
    // numbers add without rounding. Whole numbers above m0, minus infinity
    // before the first key: m the largest reference of a block, l this lane's
    // share of the sum times 2^-m; u the power of two of O, um the largest a
    // block asked for
    float m0 = 0.f, m = -INFINITY, l = 0.f, u = -INFINITY, um = -INFINITY;
    auto first = [&](float mb) {
        const float c = b1 - b0 > KG && fabsf(mb) < 256.f ? ceilf(mb * 65536.f) * 0x1p-16f : mb;
        if (m == -INFINITY && mb > -INFINITY) m0 = c;
    };
    int last = 0;
    auto pow_of = [](float d) { return (int)fmaxf(d, -1000.f); };  // of a difference, which may be of infinities

    bool any = false;  // a marked block was left out
    for (int bb = b0, it = 0; bb < b1; bb += KG, ++it) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies
        __syncthreads();  // every wave's; the other buffer's readers are done
        const int b = bb + kg, xb = __builtin_amdgcn_readfirstlane(xn), ve = (int16_t)xb, ke = (xb - ve) >> 16;
        xn = ex[min(b + KG, b1 - 1)];
        if (bb + KG < b1) copy(bb + KG, (it + 1) & 1);
        if (b >= b1) continue;  // uniform over the wave
        const uint8_t* kf = sm + ((it & 1) * KG + kg) * BB + lane * 16;
        const uint8_t* vf = kf + KS * 2048;
        f16v sh, sl;
#pragma unroll
        for (int e = 0; e < 16; ++e) sh[e] = sl[e] = 0.f;
        h8v ah[2], al[2];  // the next step's fragments are read in front of a step's products
        auto read = [&](int s) { ah[s & 1] = *(const h8v*)(kf + s * 2048), al[s & 1] = *(const h8v*)(kf + s * 2048 + 1024); };
        read(0);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            if (s + 1 < KS) read(s + 1);
            __builtin_amdgcn_sched_barrier(0);
            sh = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[s & 1], qh[s], sh, 0, 0, 0);
            sl = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[s & 1], qh[s], sl, 0, 0, 0);
            sl = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[s & 1], ql[s], sl, 0, 0, 0);
        }
        if (ve >= kPlain / 2) {
            any = true;
            continue;
        }
        // scores in log2 units; keys 8 (e / 4) + 4 h + e % 4 of the block
        const int sg = sign_of(b);
        const float c = ldexpf(sg ? -cq : cq, -ke);
        float x[16], mb = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) x[e] = (sh[e] + sl[e]) * c;
        if (b * kKB + kKB - 1 > start + t0) {  // keys past the first token's position: the causal mask
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (b * kKB + 8 * (e >> 2) + 4 * h + (e & 3) > pt) x[e] = -INFINITY;
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) mb = fmaxf(mb, x[e]);
        mb = fmaxf(mb, __shfl_xor(mb, 32, 64));
        if (__ballot(m == -INFINITY)) first(mb);
        const float rf = ceilf(mb - m0), rz = mb == -INFINITY ? 0.f : rf + m0;  // no key yet: every p is 0
        // O takes this block's power of two (its largest p near 1, times V's),
        // at most 2^60 below the largest so far: what is smaller is below
        // every rounding of the row
        const float ub = rf - (float)ve;
        um = fmaxf(um, ub);
        const float un = fmaxf(ub, um - 60.f);
        const float up = ldexpf(1.f, 14 + pow_of(ub - un)), ao = ldexpf(sg != last ? -1.f : 1.f, pow_of(u - un));
        u = un;
        last = sg;
        float lb = 0.f;
        u32x4 ph[2], pl[2];
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
            const float p0 = __builtin_amdgcn_exp2f(x[e] - rz), p1 = __builtin_amdgcn_exp2f(x[e + 1] - rz);
            lb += p0 + p1;
            uint32_t lo;
            ph[e >> 3][(e & 7) >> 1] = split2(p0 * up, p1 * up, lo);
            pl[e >> 3][(e & 7) >> 1] = lo;
        }
        const float mn = fmaxf(m, rf);
        l = ldexpf(l, pow_of(m - mn)) + ldexpf(lb, pow_of(rf - mn));
        m = mn;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            h8v vh[2], vl[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                vh[s] = *(const h8v*)(vf + (dt * 2 + s) * 2048);
                vl[s] = *(const h8v*)(vf + (dt * 2 + s) * 2048 + 1024);
            }
            f16v y;
#pragma unroll
            for (int e = 0; e < 16; ++e) y[e] = 0.f;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                y = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl[s], __builtin_bit_cast(h8v, ph[s]), y, 0, 0, 0);
                y = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[s], __builtin_bit_cast(h8v, pl[s]), y, 0, 0, 0);
            }
#pragma unroll
            for (int s = 0; s < 2; ++s)
                y = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[s], __builtin_bit_cast(h8v, ph[s]), y, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 16; ++e) o[dt][e] = __builtin_fmaf(ao, o[dt][e], y[e]);
        }
    }
    // The marked blocks, in fp32 from the cache, value after value in every
    // lane: positions a row does not see are left out, and every position is
    // added at its own power of two. After the others, where the registers of
    // the split query are free.
    for (int b = b0 + kg; any && b < b1; b += KG) {
        if ((int16_t)__builtin_amdgcn_readfirstlane(ex[b]) < kPlain / 2) continue;
        int rp = rc;
        asm volatile("" : "+v"(rp));  // the row's addresses are formed here, not held through the loop above
        const int tp = t0 + rp / R;
        const float* q = qkv + (size_t)tp * ldqkv + (size_t)(g * R + rp % R) * HD;
        const float2* cs = rope + (size_t)(start + tp) * half;
        const size_t row0 = (size_t)g * ctx;
        const int lastp = start + n_tok - 1;
        float x[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) x[e] = 0.f;
#pragma unroll 1
        for (int i = 0; i < 4; ++i) {  // positions 8 i + 4 h + 0 .. 3
            float s4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int d = 0; d < half; ++d) {
                const float2 c = cs[d];
                const float qa = rot_lo(q[d], q[half + d], c), qb = rot_hi(q[d], q[half + d], c);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float* k = kc + (row0 + min(b * kKB + 8 * i + 4 * h + j, lastp)) * HD + d;
                    s4[j] = __builtin_fmaf(qa, k[0], __builtin_fmaf(qb, k[half], s4[j]));
                }
            }
#pragma unroll
            for (int e = 0; e < 12; ++e) x[e] = x[e + 4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                x[12 + j] = b * kKB + 8 * i + 4 * h + j > pt ? -INFINITY : s4[j] * (1.4426950408889634f / sqrtf((float)HD));
        }
        float mb = -INFINITY, lb = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) mb = fmaxf(mb, x[e]);
        mb = fmaxf(mb, __shfl_xor(mb, 32, 64));
        if (__ballot(m == -INFINITY)) first(mb);
        const float rf = ceilf(mb - m0), rz = mb == -INFINITY ? 0.f : rf + m0, mn = fmaxf(m, rf);
#pragma unroll
        for (int e = 0; e < 16; ++e) lb += __builtin_amdgcn_exp2f(x[e] - rz);
        l = ldexpf(l, pow_of(m - mn)) + ldexpf(lb, pow_of(rf - mn));
        m = mn;
#pragma unroll 1
        for (int i = 0; i < 16; ++i) {
            const float own = x[0], other = __shfl_xor(own, 32, 64);
#pragma unroll
            for (int e = 0; e < 15; ++e) x[e] = x[e + 1];
#pragma unroll 1
            for (int hh = 0; hh < 2; ++hh) {
                const int key = b * kKB + 8 * (i >> 2) + 4 * hh + (i & 3);
                if (key > pt) continue;
                const float xs = hh == h ? own : other, rs = xs == -INFINITY ? 0.f : ceilf(xs - m0);
                const float ps = __builtin_amdgcn_exp2f(xs - (rs + m0));
                const float* vp = vc + (row0 + key) * HD + 4 * h;  // read twice: the registers are full
                float mv = 0.f;
#pragma unroll 1
                for (int d = 0; d < HD; d += 8) {
                    const float4 a = *(const float4*)(vp + d);
                    const float v[4] = {fabsf(a.x), fabsf(a.y), fabsf(a.z), fabsf(a.w)};
#pragma unroll
                    for (int k = 0; k < 4; ++k) mv = fmaxf(mv, v[k] <= 3.4028234e38f ? v[k] : 0.f);
                }
                const float ub = mv > 0.f && xs > -INFINITY ? rs - (float)up_exp(mv) : -INFINITY;
                um = fmaxf(um, ub);
                const float un = fmaxf(ub, um - 60.f);
                const int eo = pow_of(u - un), ev = min(pow_of(rs + 14.f - un), 1000);
                u = un;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int q4 = 0; q4 < 4; ++q4) {
                        const float4 a = *(const float4*)(vp + 32 * dt + 8 * q4);
                        const float v[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const int e = 4 * q4 + k;
                            o[dt][e] = __builtin_fmaf(last ? -ps : ps, ldexpf(v[k], ev), ldexpf(o[dt][e], eo));
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
            }
        }
    }
    l += __shfl_xor(l, 32, 64);
    const int un = min(pow_of(u - m) - 14, 1000);  // O to the units of l
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[dt][e] = ldexpf(last ? -o[dt][e] : o[dt][e], un);
    m += m0;

    // merge of the key groups, in group order
    if constexpr (KG > 1) {
        float* const om = (float*)sm;                 // [RT][HD][32 rows]
        float* const ml = om + RT * HD * 32;          // [RT][2][32]
#pragma unroll
        for (int q = 1; q < KG; ++q) {
            __syncthreads();
            if (kg == q) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        om[(rt * HD + 32 * dt + 8 * (e >> 2) + 4 * h + (e & 3)) * 32 + n] = o[dt][e];
                if (h == 0) ml[(rt * 2) * 32 + n] = m, ml[(rt * 2 + 1) * 32 + n] = l;
            }
            __syncthreads();
            if (kg == 0) {
                const float m2 = ml[(rt * 2) * 32 + n], l2 = ml[(rt * 2 + 1) * 32 + n];
                const float mn = fmaxf(m, m2), mz = mn == -INFINITY ? 0.f : mn;
                const float a1 = __builtin_amdgcn_exp2f(m - mz), a2 = __builtin_amdgcn_exp2f(m2 - mz);
                m = mn;
                l = __builtin_fmaf(l, a1, l2 * a2);
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        o[dt][e] = __builtin_fmaf(o[dt][e], a1, om[(rt * HD + 32 * dt + 8 * (e >> 2) + 4 * h + (e & 3)) * 32 + n] * a2);
            }
        }
    }
    if (kg != 0 || r >= NR) return;
    const int head = g * R + hd;
    if (nz > 1) {  // this range's O, m and l: [range][token][head][HD + 4]
        float* d = part + (((size_t)z * n_tok + t0 + ti) * n_heads + head) * (HD + 4);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *(float4*)(d + 32 * dt + 8 * q + 4 * h) = make_float4(o[dt][4 * q], o[dt][4 * q + 1], o[dt][4 * q + 2], o[dt][4 * q + 3]);
        if (h == 0) *(float4*)(d + HD) = make_float4(m, l, 0.f, 0.f);
        return;
    }
    float* d = out + (size_t)(t0 + ti) * ldo + (size_t)head * HD;
    const float il = 1.f / l;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *(float4*)(d + 32 * dt + 8 * q + 4 * h) =
                make_float4(o[dt][4 * q] * il, o[dt][4 * q + 1] * il, o[dt][4 * q + 2] * il, o[dt][4 * q + 3] * il);
}

// Merge of a row's key ranges in range order: one thread per output value.
template <int HD>
__global__ __launch_bounds__(HD) void k_attn_fa_sum(const float* part, int n_tok, int n_heads, int nz, float* out, int ldo) {
    const int t = blockIdx.x, head = blockIdx.y, d = threadIdx.x;
    const size_t zs = (size_t)n_tok * n_heads * (HD + 4);
    const float* p = part + ((size_t)t * n_heads + head) * (HD + 4);
    float m = -INFINITY;
    for (int z = 0; z < nz; ++z) m = fmaxf(m, p[z * zs + HD]);
    float o = 0.f, l = 0.f;
    for (int z = 0; z < nz; ++z) {
        const float a = __builtin_amdgcn_exp2f(p[z * zs + HD] - m);
        l = __builtin_fmaf(p[z * zs + HD + 1], a, l);
        o = __builtin_fmaf(p[z * zs + d], a, o);
    }
    out[(size_t)t * ldo + (size_t)head * HD + d] = o / l;
}

template <int HD, int RT, int KG> static size_t fa_lds() {
    return std::max<size_t>(2 * (size_t)KG * fa_block_bytes<HD>(), (size_t)RT * (HD + 2) * 32 * sizeof(float));
}

template <int HD, int RT, int KG>
static void fa_go(const FaArgs& a, const FaWork& w, int nz, float* part, hipEvent_t stop) {
    const int TB = 32 * RT / (a.n_heads / a.n_kv);
    const dim3 grid((a.n_tok + TB - 1) / TB * a.n_kv, nz);
    if (stop && nz == 1)
        hipExtLaunchKernelGGL((k_attn_fa<HD, RT, KG>), grid, dim3(64 * RT * KG), (fa_lds<HD, RT, KG>()), a.s, nullptr, stop, 0,
                              a.qkv, a.ldqkv, a.n_tok, a.n_heads, a.n_kv, a.start, a.rope, a.kc, a.vc, a.ctx, w, a.out, a.ldo, part, nz);
    else
        hipLaunchKernelGGL((k_attn_fa<HD, RT, KG>), grid, dim3(64 * RT * KG), (fa_lds<HD, RT, KG>()), a.s, a.qkv, a.ldqkv,
                           a.n_tok, a.n_heads, a.n_kv, a.start, a.rope, a.kc, a.vc, a.ctx, w, a.out, a.ldo, part, nz);
    if (nz > 1) {
        const dim3 g2(a.n_tok, a.n_heads);
        if (stop)
            hipExtLaunchKernelGGL(k_attn_fa_sum<HD>, g2, dim3(HD), 0, a.s, nullptr, stop, 0, (const float*)part, a.n_tok,
                                  a.n_heads, nz, a.out, a.ldo);
        else
            hipLaunchKernelGGL(k_attn_fa_sum<HD>, g2, dim3(HD), 0, a.s, (const float*)part, a.n_tok, a.n_heads, nz, a.out, a.ldo);
    }
}

template <int HD> static int fa_run(const FaArgs& a, uint8_t* buf, size_t cap, hipEvent_t start, hipEvent_t stop) {
    const int p_end = a.start + a.n_tok, R = a.n_heads / a.n_kv;
    FaWork w;
    w.n_blk = (p_end + kKB - 1) / kKB;
    const size_t frag = (size_t)a.n_kv * w.n_blk * fa_block_bytes<HD>();
    w.frag = buf;
    w.exps = (int*)(buf + frag);
    const size_t used = fa_bytes(HD, a.n_kv, p_end);
    const dim3 grid(w.n_blk, a.n_kv);
    if (start)
        hipExtLaunchKernelGGL(k_kv_split<HD>, grid, dim3(2 * HD), 0, a.s, start, nullptr, 0, a.qkv, a.ldqkv, a.n_heads,
                              a.n_kv, a.start, p_end, a.rope, a.kc, a.vc, a.ctx, w);
    else
        hipLaunchKernelGGL(k_kv_split<HD>, grid, dim3(2 * HD), 0, a.s, a.qkv, a.ldqkv, a.n_heads, a.n_kv, a.start, p_end,
                           a.rope, a.kc, a.vc, a.ctx, w);
    ORC_LAUNCH_CHECK();
    auto wgs = [&](int rt) { return (long)((a.n_tok + 32 * rt / R - 1) / (32 * rt / R)) * a.n_kv; };
    const int rt = wgs(4) >= g_n_cu / 2 ? 4 : wgs(2) >= g_n_cu / 2 ? 2 : 1;
    // key ranges of at least eight rounds of two blocks while CUs are idle
    int nz = (int)std::max<long>(1, std::min<long>(g_n_cu / wgs(rt), w.n_blk / 16));
    const size_t per = (size_t)a.n_tok * a.n_heads * (HD + 4) * sizeof(float);
    nz = (int)std::max<size_t>(1, std::min<size_t>(nz, (cap - used) / per));
    float* const part = (float*)(buf + used);
    if (rt == 4) fa_go<HD, 4, 2>(a, w, nz, part, stop);
    else if (rt == 2) fa_go<HD, 2, 2>(a, w, nz, part, stop);
    else fa_go<HD, 1, 2>(a, w, nz, part, stop);
    ORC_LAUNCH_CHECK();
    return ORC_OK;
}

static_assert(8 * (32768 / kKB) * (fa_block_bytes<128>() + sizeof(int)) + 256 * 32 * (128 + 4) * sizeof(float) <= kPfWorkBytes,
              "32 K positions of eight 128-wide kv heads and their key ranges");

size_t fa_bytes(int hd, int n_kv, int p_end) {
    const size_t n = (size_t)n_kv * ((p_end + kKB - 1) / kKB);
    return (n * (hd * 256 + sizeof(int)) + 255) / 256 * 256;
}

int fa_launch(int head_dim, const FaArgs& a, uint8_t* work, hipEvent_t start, hipEvent_t stop) {
    return head_dim == 64 ? fa_run<64>(a, work, kPfWorkBytes, start, stop)
                          : fa_run<128>(a, work, kPfWorkBytes, start, stop);
}

}  // namespace orc
