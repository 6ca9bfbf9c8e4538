// Dynamic per-token int8 activation quant (gfx950).
//
// Semantics follow the reference quantiser with a per-token spec
// (fakequant_lab/quant.py:89-105 group_params, :135-141 quantize_with):
//   s = bf16_rne(max|x| / 127)   -- fp32 divide, then rounded to bf16 BEFORE use
//   s = bf16 tiny (2^-126)       -- when that bf16 value is zero
//   q = clamp(rint(x / s), -128, 127), rint = round half to even, true fp32 divide
// The quotient is the IEEE divide's (the reference kernel insists on it,
// npu_ops/kernel/midgroup_quant_a.inc:55-62): a plain reciprocal multiply
// would flip half-way cases relative to torch.  The codes here come from a
// reciprocal multiply refined once (quant8_fast, common.h), which gives the
// divide's result for every input; rows whose scale is tiny, infinite or NaN
// divide per element.
//
// Layout: one workgroup per row (256 threads, 1024 for rows longer than 8192
// elements, so a decode-sized call still has enough loads in flight; long
// rows of a small batch are split over several workgroups).  The row is read
// once with 16-byte loads into registers, |x| is reduced as integers (for
// finite bf16 the magnitude order equals the order of the 15 low bits), then
// the same registers are quantised and written back as 8-byte int8 stores.
//
// Output order: plain (a_q[m, k]) or, for a ragged group geometry, the padded
// group layout the GEMM reads (kgeom.h; the reference's quantiser writes its
// activation planes in the same padded layout, midgroup_quant_a.inc:7-12):
// code k goes to (k / group) * stride + k % group, and the padding slots of
// every group are written as zero.
#include "common.h"
#include "kgeom.h"
#include "launch.h"

namespace w4a8 {
namespace {

constexpr int kThreads = 256;

// Block-wide max of a uint32 over NT threads.
template <int NT>
__device__ __forceinline__ uint32_t block_max(uint32_t v, uint32_t* red) {
    v = wave_max(v);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) v = max(v, red[w]);
    return v;
}

// Padded group layout of one row.
struct PadMap {
    int group;    // quant group
    int stride;   // ceil_to(group, 64)
    int G;        // groups
    int kpad;     // padded row length
};

__device__ __forceinline__ int pad_dst(int k, const PadMap& pm) {
    const int g = k / pm.group;
    return g * pm.stride + (k - g * pm.group);
}

// Zero the padding slots [real, stride) of every group, in units of UNIT bytes
// (real lengths are multiples of UNIT).
template <int UNIT>
__device__ __forceinline__ void zero_pads(int8_t* qr, int K, const PadMap& pm) {
    for (int u = threadIdx.x; u < pm.kpad / UNIT; u += blockDim.x) {
        const int p = u * UNIT;
        const int g = p / pm.stride;
        const int real = (g + 1 < pm.G) ? pm.group : K - (pm.G - 1) * pm.group;
        if (p - g * pm.stride >= real) {
            if constexpr (UNIT == 8) *reinterpret_cast<uint2*>(qr + p) = make_uint2(0u, 0u);
            else qr[p] = 0;
        }
    }
}

// Vector path: K % 8 == 0, rows 16-byte aligned; with PAD also group % 8 == 0
// (an 8-code unit never straddles a group).  A workgroup holds its row in
// registers as 16-byte units, unit t + i NT in thread t.  With SPLIT (long rows of
// small batches) gridDim.y workgroups share a row: each reads all of it for the
// absmax, every load in flight at once, and quantises the units of i = blockIdx.y,
// so the per-element work spreads over gridDim.y CUs.  Rows past VPT * NT units
// (SPLIT only) are read in a loop instead, and the workgroup's own units again.
//
// Bound by memory on many rows (16384 x 27648: 253 -> 229 us, 5.9 TB/s of its 1.36
// GB, from six instead of fourteen vector instructions per element) and by
// latency on few: one memory round trip, two block-wide steps and the per-element
// work of a thread's units (1 x 5120 3.1 -> 2.5 us in a graph of back-to-back calls).
template <int VPT, int NT, bool PAD, bool SPLIT>
__global__ __launch_bounds__(NT) void quant_act_vec_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int8_t* __restrict__ aq, int64_t lda,
    uint16_t* __restrict__ ascale, int K, const PadMap pm) {
    __shared__ uint32_t red[NT / 64];
    const int64_t row = blockIdx.x;
    // buffer loads (units past the row read zero): under a branch each load is
    // followed by register copies that wait for it before the next is issued
    const auto xr = make_rsrc(x + row * ldx, static_cast<uint32_t>(K) * 2u);
    const int nvec = K >> 3;
    const int own = SPLIT ? static_cast<int>(blockIdx.y) : 0;
    auto unit = [&](int i) { return buf_load16(xr, (threadIdx.x + static_cast<uint32_t>(i) * NT) * 16u); };
    uint4 v[VPT];
    uint32_t amax = 0u;
    if (SPLIT && static_cast<int>(gridDim.y) > VPT) {
        // eight loads in flight for a few rows (VPT = 8); one at a time past 16 rows, where
        // the workgroups of a CU hide each other's latency (40960 x 64 rows 4.8 us against 5.4)
        constexpr int U = VPT == 8 ? 8 : 1;
        const uint4 w = unit(own);
        for (int i0 = 0; i0 < static_cast<int>(gridDim.y); i0 += U) {
#pragma unroll
            for (int i = 0; i < U; ++i) v[i] = unit(i0 + i);
#pragma unroll
            for (int i = 0; i < U; ++i) amax = max(amax, abs_bits_max8(v[i]));
        }
        v[0] = w;
    } else {
#pragma unroll
        for (int i = 0; i < VPT; ++i) v[i] = unit(i);
#pragma unroll
        for (int i = 0; i < VPT; ++i) amax = max(amax, abs_bits_max8(v[i]));
        if constexpr (SPLIT) {
            uint4 w = v[0];
#pragma unroll
            for (int i = 1; i < VPT; ++i)
                if (i == own) w = v[i];
            v[0] = w;
        }
    }
    amax = block_max<NT>(amax, red);
    const uint32_t sbits = scale_from_amax(amax);
    const RowScale q = row_scale(bf16_bits_to_f32(sbits));
    const bool first = own == 0;
    if (threadIdx.x == 0 && first) ascale[row] = static_cast<uint16_t>(sbits);
    int8_t* qr = aq + row * lda;
#pragma unroll
    for (int i = 0; i < (SPLIT ? 1 : VPT); ++i) {
        const int idx = static_cast<int>(threadIdx.x) + (SPLIT ? own : i) * NT;
        const uint2 o = quant_unit(v[i], q);
        if (idx < nvec) *reinterpret_cast<uint2*>(qr + (PAD ? pad_dst(idx * 8, pm) : idx * 8)) = o;
    }
    if constexpr (PAD) {
        if (first) zero_pads<8>(qr, K, pm);
    }
}

// General path: any K and strides; two passes over the row (the second one
// hits cache).
__global__ __launch_bounds__(kThreads) void quant_act_scalar_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, int8_t* __restrict__ aq, int64_t lda,
    uint16_t* __restrict__ ascale, int K, bool pad, const PadMap pm) {
    __shared__ uint32_t red[4];
    const int64_t row = blockIdx.x;
    const uint16_t* xr = x + row * ldx;
    uint32_t amax = 0u;
    for (int k = threadIdx.x; k < K; k += kThreads) amax = max(amax, static_cast<uint32_t>(xr[k]) & 0x7fffu);
    amax = block_max<kThreads>(amax, red);
    const uint32_t sbits = scale_from_amax(amax);
    const float s = bf16_bits_to_f32(sbits);
    if (threadIdx.x == 0) ascale[row] = static_cast<uint16_t>(sbits);
    int8_t* qr = aq + row * lda;
    for (int k = threadIdx.x; k < K; k += kThreads)
        qr[pad ? pad_dst(k, pm) : k] = static_cast<int8_t>(quant_div(bf16_bits_to_f32(xr[k]), s));
    if (pad) zero_pads<1>(qr, K, pm);
}

}  // namespace

hipError_t launch_quant_act(const uint16_t* x, int64_t ldx, int8_t* a_q, int64_t lda,
                            uint16_t* a_scale, int64_t M, int64_t K, int64_t group, hipStream_t stream) {
    if (M == 0) return hipSuccess;
    const dim3 grid(static_cast<unsigned>(M));
    const dim3 block(kThreads);
    const bool pad = group > 0 && !geom::is_unpadded(K, group);
    PadMap pm{};
    if (pad) {
        pm.group = static_cast<int>(group);
        pm.stride = static_cast<int>(geom::group_stride(group));
        pm.G = static_cast<int>(geom::num_groups(K, group));
        pm.kpad = static_cast<int>(geom::kpad(K, group));
    }
    const bool aligned = (K % 8 == 0) && (ldx % 8 == 0) && (lda % 8 == 0) && (!pad || group % 8 == 0) &&
                         (reinterpret_cast<uintptr_t>(x) % 16 == 0) &&
                         (reinterpret_cast<uintptr_t>(a_q) % 8 == 0);
    const int64_t nvec = K / 8;
    const int iK = static_cast<int>(K);
    // Rows of up to 8192 elements: 256 threads.  Longer rows of a small batch
    // (M < 256, too few rows to fill the GPU) are split: over 512-thread workgroups
    // of one 16-byte unit per thread up to 16 rows, 1024-thread ones past them
    // (K = 27648, us: 16 rows 3.2 / 3.3, 64 rows 4.1 / 3.7, 200 rows 7.2 / 6.8) and for
    // rows past 32768 elements, which 512 threads no longer hold (131072: one row
    // 6.9 us / 4.7, 16 rows 7.5 / 5.5, each against the better loop).
    // Longer rows otherwise: 1024 threads per row.
    const bool vec = aligned && K < (int64_t{1} << 30);   // rows in 32-bit buffer offsets
    if (vec && nvec > 4 * kThreads && M < 256) {
        const int nt = M <= 16 && nvec <= 8 * 512 ? 512 : 1024;
        const dim3 g2(static_cast<unsigned>(M), static_cast<unsigned>((nvec + nt - 1) / nt));
#define W4A8_QSPLIT(V, NT)                                                                                     \
    if (pad) quant_act_vec_kernel<V, NT, true, true><<<g2, dim3(NT), 0, stream>>>(x, ldx, a_q, lda, a_scale, iK, pm); \
    else quant_act_vec_kernel<V, NT, false, true><<<g2, dim3(NT), 0, stream>>>(x, ldx, a_q, lda, a_scale, iK, pm);
        if (nt == 512) { W4A8_QSPLIT(8, 512) }
        else if (M <= 16) { W4A8_QSPLIT(8, 1024) }
        else { W4A8_QSPLIT(4, 1024) }
#undef W4A8_QSPLIT
        return hipGetLastError();
    }
    int vpt = 0;
    const bool wide = nvec > 4 * kThreads;
    const int nt = wide ? 4 * kThreads : kThreads;
    for (int v : {1, 2, 4, 8})
        if (vpt == 0 && vec && nvec <= v * nt) vpt = v;
#define W4A8_QVEC(V, NT)                                                                                      \
    if (pad) quant_act_vec_kernel<V, NT, true, false><<<grid, dim3(NT), 0, stream>>>(x, ldx, a_q, lda, a_scale, iK, pm); \
    else quant_act_vec_kernel<V, NT, false, false><<<grid, dim3(NT), 0, stream>>>(x, ldx, a_q, lda, a_scale, iK, pm);
    if (vpt == 0) {
        quant_act_scalar_kernel<<<grid, block, 0, stream>>>(x, ldx, a_q, lda, a_scale, iK, pad, pm);
    } else if (!wide) {
        if (vpt == 1) { W4A8_QVEC(1, kThreads) }
        else if (vpt == 2) { W4A8_QVEC(2, kThreads) }
        else { W4A8_QVEC(4, kThreads) }
    } else {
        if (vpt == 1) { W4A8_QVEC(1, 4 * kThreads) }
        else if (vpt == 2) { W4A8_QVEC(2, 4 * kThreads) }
        else if (vpt == 4) { W4A8_QVEC(4, 4 * kThreads) }
        else { W4A8_QVEC(8, 4 * kThreads) }
    }
#undef W4A8_QVEC
    return hipGetLastError();
}

}  // namespace w4a8
