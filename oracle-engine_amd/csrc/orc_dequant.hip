// Bit-exact dequant codecs and the embedding-row gather (gfx950).
//
// Replaces the block codecs and dequantize_row / dequantize_into of the
// reference (core/gguf_parser.cpp:420-482, 1002-1154) and the embedding
// lookups of Model::forward / forward_prefill (core/model.cpp:349-358, 549-558).
#include "orc_internal.hpp"

// ── bit-exact dequant (core/gguf_parser.cpp:1029-1154) ───────────────────────
namespace orc {
// One thread per eight consecutive output values (octet j of 32-value group
// g); rounding exactly as the reference build: Q4_0/Q8_0/F16/BF16 one product
// or exact conversion, Q4_K fma(d*sc, q, -(dmin*m)) (the reference's d1*q - m1f
// contracts to one FMA), Q6_K (d*sc)*q with two roundings. Every load is whole
// and independent of the others: a row's gather is one memory round trip after
// its id. With one thread per 32 values and a load per byte a 3072-value Q6_K
// row took 13.8 us (7% of the passes of a 4-block decode step); now 4.0.
__device__ __forceinline__ uint32_t byte_of(u32x2 v, int i) { return ((i < 4 ? v.x : v.y) >> (8 * (i & 3))) & 0xFFu; }

__device__ __forceinline__ void dequant8(int type, const uint8_t* w, int64_t g, int j, float (&out)[8]) {
    switch (type) {
        case ORC_F32: {
            const uint8_t* p = w + g * 128 + 32 * j;
            const u32x4 a = ld16(p), b = ld16(p + 16);
            const uint32_t q[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] = __builtin_bit_cast(float, q[i]);
            break;
        }
        case ORC_F16:
        case ORC_BF16: {  // BF16: the high half of an fp32 (core/gguf_parser.cpp:1034-1040)
            const u32x4 a = ld16(w + g * 64 + 16 * j);
            const uint32_t q[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t v = (q[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
                out[i] = type == ORC_F16 ? h2f(v) : __builtin_bit_cast(float, v << 16);
            }
            break;
        }
        case ORC_Q8_0:
        case ORC_Q8_0_X8: {  // X8: block g&7 of the 272-byte group g>>3: scale at 2*(g&7), codes at 16+32*(g&7)
            const uint8_t* grp = w + (g >> 3) * 272;
            const uint8_t* pd = type == ORC_Q8_0 ? w + g * 34 : grp + 2 * (g & 7);
            const uint8_t* pq = type == ORC_Q8_0 ? w + g * 34 + 2 : grp + 16 + 32 * (g & 7);
            const u32x2 q = ld8(pq + 8 * j);
            const float d = h2f(ld2(pd));
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] = d * (float)(int8_t)byte_of(q, i);
            break;
        }
        case ORC_Q4_0: {  // values 0-15 low nibbles, 16-31 high nibbles
            const uint8_t* b = w + g * 18;
            const u32x2 q = ld8(b + 2 + 8 * (j & 1));
            const float d = h2f(ld2(b));
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] = d * (float)((int)((byte_of(q, i) >> (4 * (j >> 1))) & 0xF) - 8);
            break;
        }
        case ORC_Q4_K: {  // 32 values = one sub-block
            const int s = (int)(g & 7);
            const uint8_t* b = w + (g >> 3) * 144;
            const u32x4 hdr = ld16(b);
            const u32x2 q = ld8(b + 16 + 32 * (s >> 1) + 8 * j);
            uint32_t sc, mn;
            q4k_scale_min(s, hdr.y, hdr.z, hdr.w, sc, mn);
            const float d1 = h2f(hdr.x & 0xFFFFu) * (float)sc, m1 = h2f(hdr.x >> 16) * (float)mn;
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] = __builtin_fmaf(d1, (float)((byte_of(q, i) >> (4 * (s & 1))) & 0xF), -m1);
            break;
        }
        case ORC_Q6_K: {  // 32 values = values 128hh+32gg+[0,32) of superblock g>>3
            const uint8_t* b = w + (g >> 3) * 210;
            const int s = (int)(g & 7), hh = s >> 2, gg = s & 3;
            const u32x2 ql = ld8(b + 64 * hh + 32 * (gg & 1) + 8 * j), qh = ld8(b + 128 + 32 * hh + 8 * j);
            const int8_t sc = (int8_t)b[192 + 8 * hh + 2 * gg + (j >> 1)];
            const float ds = h2f(ld2(b + 208)) * (float)sc;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int q = (int)(((byte_of(ql, i) >> (4 * (gg >> 1))) & 0xF) | (((byte_of(qh, i) >> (2 * gg)) & 3) << 4));
                out[i] = ds * (float)(q - 32);
            }
            break;
        }
    }
}

__global__ void k_dequant(int type, const uint8_t* w, int64_t n_oct, float* y) {
    const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= n_oct) return;
    float v[8];
    dequant8(type, w, o >> 2, (int)(o & 3), v);
    float4* d = (float4*)(y + o * 8);
    d[0] = make_float4(v[0], v[1], v[2], v[3]);
    d[1] = make_float4(v[4], v[5], v[6], v[7]);
}

__global__ void k_embed(int type, const uint8_t* table, int n_in, int n_rows, uint64_t row_bytes, const int32_t* ids,
                        float* y, int ldy) {
    const int t = blockIdx.y;
    const int o = blockIdx.x * blockDim.x + threadIdx.x;
    if (o * 8 >= n_in) return;
    int id = ids[t];
    if (id < 0 || id >= n_rows) id = 0;
    float v[8];
    dequant8(type, table + (uint64_t)id * row_bytes, o >> 2, o & 3, v);
    float4* d = (float4*)(y + (size_t)t * ldy + o * 8);
    d[0] = make_float4(v[0], v[1], v[2], v[3]);
    d[1] = make_float4(v[4], v[5], v[6], v[7]);
}
}  // namespace orc

using namespace orc;

static bool dq_type_ok(int t) {
    return t == ORC_F32 || t == ORC_F16 || t == ORC_BF16 || t == ORC_Q4_0 || t == ORC_Q8_0 || t == ORC_Q4_K ||
           t == ORC_Q6_K;
}

extern "C" int orc_dequant(int type, const void* d_w, int64_t n_el, float* d_y, orc_stream_t stream) {
    if (!initialized()) return set_error(ORC_E_NOINIT, "orc_init not called");
    if (!dq_type_ok(type) && type != ORC_Q8_0_X8)
        return set_error(ORC_E_UNSUPPORTED, "dequant: unsupported type " + std::to_string(type));
    const int be = (type == ORC_Q4_K || type == ORC_Q6_K || type == ORC_Q8_0_X8) ? 256 : 32;
    if (n_el <= 0 || n_el % be || !d_w || !d_y) return set_error(ORC_E_INVALID, "dequant: bad size or pointer");
    if ((uintptr_t)d_y & 15) return set_error(ORC_E_INVALID, "dequant: output must be 16-byte aligned");
    const int64_t octets = n_el / 8;
    hipLaunchKernelGGL(k_dequant, dim3((unsigned)((octets + 255) / 256)), dim3(256), 0, resolve_stream(stream), type,
                       (const uint8_t*)d_w, octets, d_y);
    ORC_LAUNCH_CHECK();
    return ORC_OK;
}

extern "C" int orc_embed(int type, const void* d_table, int n_in, int n_rows, const int32_t* d_ids, int n_tok,
                         float* d_y, int ldy, orc_stream_t stream) {
    if (!initialized()) return set_error(ORC_E_NOINIT, "orc_init not called");
    if (!dq_type_ok(type)) return set_error(ORC_E_UNSUPPORTED, "embed: unsupported type " + std::to_string(type));
    const int be = (type == ORC_Q4_K || type == ORC_Q6_K) ? 256 : 32;
    if (n_in <= 0 || n_in % be || n_rows <= 0 || n_tok < 0 || ldy < n_in || ldy % 4 || !d_table || !d_ids || !d_y)
        return set_error(ORC_E_INVALID, "embed: bad arguments");
    if (n_tok == 0) return ORC_OK;
    const int octets = n_in / 8;
    hipLaunchKernelGGL(k_embed, dim3((octets + 127) / 128, n_tok), dim3(128), 0, resolve_stream(stream), type,
                       (const uint8_t*)d_table, n_in, n_rows, (uint64_t)orc_row_bytes(type, n_in), d_ids, d_y, ldy);
    ORC_LAUNCH_CHECK();
    return ORC_OK;
}
