// Rotary embedding of q and k fused with the KV-cache append (gfx950).
//
// One launch for what the decoder layer otherwise runs as a dozen elementwise
// kernels per projection output (float casts, four products, a difference, a
// sum, a concatenation, a bf16 cast for q and again for k, then an indexed
// copy into each cache).  For token t of sequence b at position p = pos[0] + t
// and pair index i < D/2 of head h (rotate-half form, x1 = x[i], x2 = x[i+D/2],
// c = cos[p, i], s = sin[p, i] in fp32):
//   y[i]       = bf16( fl(x1 * c) - fl(x2 * s) )
//   y[i + D/2] = bf16( fl(x2 * c) + fl(x1 * s) )
// each product and the sum rounded to fp32 separately (no fused multiply-add),
// then round-to-nearest-even -- the sequence torch evaluates for
// `cat([x1*c - x2*s, x2*c + x1*s]).to(bfloat16)` on float tensors.  An
// optional projection bias is added first, x = bf16(x + bias), as torch adds
// two bf16 tensors (q, k and v alike).  The q heads
// go to q_out [B, T, H, D]; the k heads to k_cache[b, h, :, p] and the raw v
// heads to v_cache[b, h, p, :] through per-dimension strides, so either cache
// layout ([B, KVH, D, L] or [B, KVH, L, D]) is served.  The position is read
// on the device, so a captured decode step advances with it; a token whose
// position falls outside [0, L) writes nothing to the caches and zeros to q.
#include "common.h"
#include "launch.h"

namespace w4a8 {
namespace {

// Workgroup (token, head): heads 0 .. H-1 are q, H .. H+KVH-1 are k (both
// rotated, one pair per thread), the rest v (two elements per thread).
__global__ __launch_bounds__(64) void rope_kv_kernel(const RopeKvArgs a) {
#pragma clang fp contract(off)
    const int tok = static_cast<int>(blockIdx.x);      // b * T + t
    const int hh = static_cast<int>(blockIdx.y);
    const int b = tok / a.T;
    const int t = tok - b * a.T;
    const int64_t p = a.pos[0] + t;
    const int half = a.D / 2;
    const bool inside = p >= 0 && p < a.L;
    const uint16_t* x = a.qkv + static_cast<int64_t>(tok) * a.ldq + hh * a.D;
    const uint16_t* bias = a.bias ? a.bias + hh * a.D : nullptr;
    // x (+ bias, rounded to bf16 as a bf16 add rounds it)
    auto in = [&](int d) {
        const float v = bf16_bits_to_f32(x[d]);
        return bias ? bf16_bits_to_f32(f32_to_bf16_bits(v + bf16_bits_to_f32(bias[d]))) : v;
    };
    if (hh >= a.H + a.KVH) {
        if (!inside) return;
        uint16_t* vr = a.v_cache + b * a.vs[0] + (hh - a.H - a.KVH) * a.vs[1] + p * a.vs[2];
        for (int d = threadIdx.x; d < a.D; d += blockDim.x)
            vr[d * a.vs[3]] = static_cast<uint16_t>(f32_to_bf16_bits(in(d)));
        return;
    }
    for (int i = threadIdx.x; i < half; i += blockDim.x) {
        uint16_t o1 = 0, o2 = 0;   // no angle row and no cache slot: q reads as zero
        if (inside) {
            const float x1 = in(i), x2 = in(i + half);
            const float c = a.cos[p * a.ldc + i], s = a.sin[p * a.ldc + i];
            const float y1 = x1 * c - x2 * s;
            const float y2 = x2 * c + x1 * s;
            o1 = static_cast<uint16_t>(f32_to_bf16_bits(y1));
            o2 = static_cast<uint16_t>(f32_to_bf16_bits(y2));
        }
        if (hh < a.H) {
            uint16_t* q = a.q_out + (static_cast<int64_t>(tok) * a.H + hh) * a.D;
            q[i] = o1;
            q[i + half] = o2;
        } else if (inside) {
            uint16_t* k = a.k_cache + b * a.ks[0] + (hh - a.H) * a.ks[1] + p * a.ks[3];
            k[i * a.ks[2]] = o1;
            k[(i + half) * a.ks[2]] = o2;
        }
    }
}

// Prefill (many tokens per sequence) on the decoder's cache layouts: K with its
// dimensions contiguous ([B, KVH, L, D] rows), V transposed (positions
// contiguous).  The kernel above writes V element by element, one cache line
// each, and works on 2 bytes per lane; here the first nqk workgroups rotate eight
// pairs per thread with 16-byte loads and stores, and the others take 64 tokens
// of one v head through LDS, so every store covers consecutive positions.  The
// same operations per element, so the same bits.  Bound by memory: 1024 tokens of
// 40 + 16 heads of 128 (29 MB) 26.1 -> 8.8 us,
// 8 sequences of them 167 -> 40.
constexpr int kRopeTile = 64;   // tokens per v workgroup

// Two packed bf16 (+ two bias elements, rounded as bf16 adds).
__device__ __forceinline__ uint32_t add_bias2(uint32_t x, uint32_t b, bool has) {
    if (!has) return x;
    return f32x2_to_bf16x2_bits(__uint_as_float(x << 16) + __uint_as_float(b << 16),
                                __uint_as_float(x & 0xffff0000u) + __uint_as_float(b & 0xffff0000u));
}

__device__ __forceinline__ uint4 load_bias(const uint16_t* bias, int off) {
    return bias ? *reinterpret_cast<const uint4*>(bias + off) : make_uint4(0u, 0u, 0u, 0u);
}

__global__ __launch_bounds__(256) void rope_kv_prefill_kernel(const RopeKvArgs a, int nqk, int tiles) {
#pragma clang fp contract(off)
    extern __shared__ uint16_t vt[];   // v workgroups: [kRopeTile][D + 2]
    const int tid = static_cast<int>(threadIdx.x);
    const int half = a.D / 2;
    const int64_t pos0 = a.pos[0];
    if (static_cast<int>(blockIdx.x) < nqk) {
        const int upr = half / 8;                          // units of eight pairs per head
        const int64_t u = static_cast<int64_t>(blockIdx.x) * 256 + tid;
        const int64_t per_tok = static_cast<int64_t>(a.H + a.KVH) * upr;
        const int64_t tok = u / per_tok;
        if (tok >= static_cast<int64_t>(a.B) * a.T) return;
        const int r = static_cast<int>(u - tok * per_tok);
        const int hh = r / upr, i0 = (r - hh * upr) * 8;
        const int b = static_cast<int>(tok / a.T);
        const int64_t p = pos0 + (tok - static_cast<int64_t>(b) * a.T);
        const bool inside = p >= 0 && p < a.L;
        uint4 o1 = make_uint4(0u, 0u, 0u, 0u), o2 = o1;    // no angle row: q reads as zero
        if (inside) {
            const uint16_t* x = a.qkv + tok * a.ldq + hh * a.D + i0;
            const uint4 v1 = *reinterpret_cast<const uint4*>(x), v2 = *reinterpret_cast<const uint4*>(x + half);
            const uint4 b1 = load_bias(a.bias, hh * a.D + i0), b2 = load_bias(a.bias, hh * a.D + i0 + half);
            const float4* cp = reinterpret_cast<const float4*>(a.cos + p * a.ldc + i0);
            const float4* sp = reinterpret_cast<const float4*>(a.sin + p * a.ldc + i0);
            const float4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
            const float c[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
            const float s[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
            const uint32_t w1[4] = {v1.x, v1.y, v1.z, v1.w}, w2[4] = {v2.x, v2.y, v2.z, v2.w};
            const uint32_t e1[4] = {b1.x, b1.y, b1.z, b1.w}, e2[4] = {b2.x, b2.y, b2.z, b2.w};
            uint32_t r1[4], r2[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const uint32_t m1 = add_bias2(w1[d], e1[d], a.bias != nullptr);
                const uint32_t m2 = add_bias2(w2[d], e2[d], a.bias != nullptr);
                const float x1 = __uint_as_float(m1 << 16), y1 = __uint_as_float(m1 & 0xffff0000u);
                const float x2 = __uint_as_float(m2 << 16), y2 = __uint_as_float(m2 & 0xffff0000u);
                const float ca = c[2 * d], cb = c[2 * d + 1], sa = s[2 * d], sb = s[2 * d + 1];
                r1[d] = f32x2_to_bf16x2_bits(x1 * ca - x2 * sa, y1 * cb - y2 * sb);
                r2[d] = f32x2_to_bf16x2_bits(x2 * ca + x1 * sa, y2 * cb + y1 * sb);
            }
            o1 = make_uint4(r1[0], r1[1], r1[2], r1[3]);
            o2 = make_uint4(r2[0], r2[1], r2[2], r2[3]);
        }
        uint16_t* o;
        if (hh < a.H) o = a.q_out + (tok * a.H + hh) * a.D + i0;
        else if (inside) o = a.k_cache + b * a.ks[0] + (hh - a.H) * a.ks[1] + p * a.ks[3] + i0;
        else return;
        *reinterpret_cast<uint4*>(o) = o1;
        *reinterpret_cast<uint4*>(o + half) = o2;
        return;
    }
    // v: tokens t0 .. t0 + 63 of sequence b, head h
    const int w = static_cast<int>(blockIdx.x) - nqk;
    const int h = w % a.KVH, bt = w / a.KVH;
    const int b = bt / tiles, t0 = (bt - b * tiles) * kRopeTile;
    const int nt = min(kRopeTile, a.T - t0);
    const int ls = a.D + 2, upr = a.D / 8;
    const int vo = (a.H + a.KVH + h) * a.D;
    for (int u = tid; u < nt * upr; u += 256) {
        const int t = u / upr, d0 = (u - t * upr) * 8;
        const uint4 v = *reinterpret_cast<const uint4*>(a.qkv + (static_cast<int64_t>(b) * a.T + t0 + t) * a.ldq + vo + d0);
        const uint4 e = load_bias(a.bias, vo + d0);
        uint32_t* l = reinterpret_cast<uint32_t*>(vt + t * ls + d0);
        l[0] = add_bias2(v.x, e.x, a.bias != nullptr);
        l[1] = add_bias2(v.y, e.y, a.bias != nullptr);
        l[2] = add_bias2(v.z, e.z, a.bias != nullptr);
        l[3] = add_bias2(v.w, e.w, a.bias != nullptr);
    }
    __syncthreads();
    const int t = tid & (kRopeTile - 1);
    const int64_t p = pos0 + t0 + t;
    if (t >= nt || p < 0 || p >= a.L) return;
    uint16_t* vr = a.v_cache + b * a.vs[0] + h * a.vs[1] + p;
    for (int d = tid / kRopeTile; d < a.D; d += 256 / kRopeTile) vr[d * a.vs[3]] = vt[t * ls + d];
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// The prefill kernel's layouts: 16-byte rows everywhere it loads or stores 16 bytes,
// K dimensions contiguous, V positions contiguous, and its v tile inside 64 KB of LDS.
bool prefill_layout(const RopeKvArgs& a) {
    return a.D % 16 == 0 && a.D <= 256 && a.ldq % 8 == 0 && a.ldc % 4 == 0 && a.ks[2] == 1 && a.ks[0] % 8 == 0 &&
           a.ks[1] % 8 == 0 && a.ks[3] % 8 == 0 && a.vs[2] == 1 && aligned16(a.qkv) &&
           (a.bias == nullptr || aligned16(a.bias)) && aligned16(a.cos) && aligned16(a.sin) && aligned16(a.q_out) &&
           aligned16(a.k_cache);
}

}  // namespace

hipError_t launch_rope_kv(const RopeKvArgs& a, hipStream_t stream) {
    const int64_t tokens = static_cast<int64_t>(a.B) * a.T;
    if (tokens <= 0) return hipSuccess;
    // The kernel above is one wave per (token, head).  Up to about twenty waves a CU they
    // are all resident and it is the quicker; past that, with a quarter of a v tile or more
    // per sequence, the prefill kernel (us, above / this one: 40 + 16 heads x 64 tokens
    // 4.2 / 4.5, x 128 5.6 / 5.0, x 256 8.5 / 5.2; 10 + 4 heads x 128 tokens 3.7 / 4.5, x 256
    // 4.3 / 4.7, x 400 5.2 / 4.7; 32 + 16 heads of 64 x 80 tokens 4.3 / 3.9).  A decode step
    // has one token per sequence.
    const int64_t waves = tokens * (a.H + 2 * a.KVH);
    const int tiles = (a.T + kRopeTile - 1) / kRopeTile;
    const int64_t nqk = (tokens * (a.H + a.KVH) * (a.D / 16) + 255) / 256;
    const int64_t nwg = nqk + static_cast<int64_t>(a.B) * tiles * a.KVH;
    if (a.T >= kRopeTile / 4 && waves >= 20 * device_cu_count() && prefill_layout(a) && nwg < (int64_t{1} << 31)) {
        const size_t lds = static_cast<size_t>(kRopeTile) * (a.D + 2) * 2;
        rope_kv_prefill_kernel<<<dim3(static_cast<unsigned>(nwg)), dim3(256), lds, stream>>>(
            a, static_cast<int>(nqk), tiles);
        return hipGetLastError();
    }
    rope_kv_kernel<<<dim3(static_cast<unsigned>(tokens), static_cast<unsigned>(a.H + 2 * a.KVH)), dim3(64), 0,
                     stream>>>(a);
    return hipGetLastError();
}

}  // namespace w4a8
