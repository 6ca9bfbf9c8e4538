// The hot torch.ops.npu.* kernels in C++: argument checks, output allocation and
// the C ABI call, without Python between the dispatcher and the launch.
//
// An op called from Python used to spend 15-25 us in its Python kernel (checks,
// three tensor allocations, ctypes), more than the launches of a decode-sized
// linear take on the GPU; here the same steps take 3-5 us (one row of a 5120 x 5120
// linear module 22 -> 7.7 us per call, the GPU's share 7.4).
//
// Schemas, fake kernels and the remaining ops stay in ops.py, the checks and their
// messages are those of the Python kernels these replace (TORCH_CHECK raises
// RuntimeError).  The C ABI library is not linked: its entry points are asked for
// once, at the first call, through the Python loader (_abi.lib(), which honours
// W4A8_AMD_LIB and raises FileNotFoundError where the library is missing), and
// workspaces come from ops._workspace, which keeps one per device and stream and
// per graph capture.
#define __HIP_PLATFORM_AMD__ 1
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>

#include <atomic>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/w4a8_amd.h"
#include "kgeom.h"

namespace {

namespace geom = w4a8::geom;
using at::Tensor;

// The C ABI entry points used here, in the order bind() receives their addresses.
#define W4A8_TORCH_FNS(F)                                                                                     \
    F(w4a8_last_error) F(w4a8_quant_act) F(w4a8_gemm_workspace_bytes) F(w4a8_gemm) F(w4a8_gemm_swiglu)        \
    F(w4a8_linear_bias) F(w4a8_rmsnorm_quant) F(w4a8_rope_kv) F(w4a8_attention) F(w4a8_attention_rope)        \
    F(w4a8_attention_workspace_bytes) F(w4a8_midgroup_quant_a) F(w4a8_midgroup_gemm_workspace_bytes)          \
    F(w4a8_midgroup_split_workspace_bytes) F(w4a8_midgroup_gemm_split) F(w4a8_midgroup_tiles_bytes)           \
    F(w4a8_midgroup_gemm_ws) F(w4a8_midgroup_gemm_tiled)

struct Abi {
#define W4A8_DECL(n) decltype(&::n) n;
    W4A8_TORCH_FNS(W4A8_DECL)
#undef W4A8_DECL
};

std::vector<std::string> abi_names() {
    return {
#define W4A8_NAME(n) #n,
        W4A8_TORCH_FNS(W4A8_NAME)
#undef W4A8_NAME
    };
}

// Set once from Python at import; never destroyed (the interpreter may be gone first).
PyObject* g_loader = nullptr;      // () -> addresses of abi_names()
PyObject* g_workspace = nullptr;   // (device index, bytes) -> (address, bytes)
Abi g_abi;
std::atomic<bool> g_bound{false};

const Abi& abi() {
    if (!g_bound.load(std::memory_order_acquire)) {
        py::gil_scoped_acquire gil;   // also serialises the first calls of several threads
        if (!g_bound.load(std::memory_order_relaxed)) {
            TORCH_CHECK(g_loader != nullptr, "w4a8: the torch layer is not initialised");
            const auto a = py::reinterpret_borrow<py::object>(g_loader)().cast<std::vector<uintptr_t>>();
            size_t i = 0;
#define W4A8_SET(n) g_abi.n = reinterpret_cast<decltype(&::n)>(a.at(i++));
            W4A8_TORCH_FNS(W4A8_SET)
#undef W4A8_SET
            g_bound.store(true, std::memory_order_release);
        }
    }
    return g_abi;
}

void check(int status, const char* what) {
    if (status == 0) return;
    static const char* const names[] = {"OK", "NULL", "SHAPE", "DTYPE", "ALIGN", "UNSUPPORTED", "WORKSPACE", "HIP"};
    const std::string name = status > 0 && status < 8 ? names[status] : std::to_string(status);
    TORCH_CHECK(false, what, " failed (", name, "): ", abi().w4a8_last_error());
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

struct Workspace {
    void* ptr = nullptr;
    int64_t bytes = 0;
};

Workspace workspace(const Tensor& t, int64_t need) {
    py::gil_scoped_acquire gil;
    const auto r = py::reinterpret_borrow<py::object>(g_workspace)(static_cast<int>(t.device().index()), need)
                       .cast<std::pair<uintptr_t, int64_t>>();
    return {reinterpret_cast<void*>(r.first), r.second};
}

Tensor empty(at::IntArrayRef sizes, at::ScalarType dt, const Tensor& like) {
    return at::empty(sizes, at::TensorOptions().dtype(dt).device(like.device()));
}

// A tensor whose rows are contiguous (and row starts a multiple of `align` elements apart).
Tensor rows(const Tensor& t, int64_t align = 1) {
    return t.stride(1) != 1 || t.stride(0) % align ? t.contiguous() : t;
}

const void* opt_ptr(const std::optional<Tensor>& t) { return t.has_value() ? t->data_ptr() : nullptr; }

bool is_scale(at::ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }
int scale_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? W4A8_DT_BF16 : W4A8_DT_F16; }

// Python's floor-based integer arithmetic is not needed: K and group are checked positive
// where the geometry divides by them.
void check_geometry(const char* op, int64_t K, int64_t group) {
    TORCH_CHECK(K > 0 && group > 0, op, ": K=", K, " and group=", group, " must be > 0");
}

int64_t quant_width(int64_t K, int64_t group) { return group > 0 && K > 0 ? geom::kpad(K, group) : K; }

// ------------------------------------------------------------------ quant
std::tuple<Tensor, Tensor> quant_pertoken(const Tensor& x0, int64_t group) {
    TORCH_CHECK(x0.dim() == 2, "w4a8_quant_pertoken: x must be [M, K]");
    TORCH_CHECK(x0.scalar_type() == at::kBFloat16, "w4a8_quant_pertoken: x must be bfloat16");
    TORCH_CHECK(group >= 0, "w4a8_quant_pertoken: group must be >= 0");
    const Tensor x = rows(x0);
    const int64_t M = x.size(0), K = x.size(1), width = quant_width(K, group);
    Tensor a_q = empty({M, width}, at::kChar, x), a_scale = empty({M}, at::kBFloat16, x);
    if (M)
        check(abi().w4a8_quant_act(x.data_ptr(), x.stride(0), a_q.data_ptr(), width, a_scale.data_ptr(), M, K, group,
                                   stream_of(x)),
              "w4a8_quant_pertoken");
    return {a_q, a_scale};
}

// ------------------------------------------------------------------ gemm
void check_weights(const Tensor& w_tiles, const Tensor& s_tiles, int64_t N, int64_t K, int64_t group) {
    TORCH_CHECK(w_tiles.scalar_type() == at::kByte &&
                    w_tiles.numel() == geom::col_blocks(N) * geom::k_tiles(K, group) * geom::kTileBytes,
                "w4a8_gemm: w_tiles must be the uint8 output of w4a8_repack for (N, K, group)");
    TORCH_CHECK(is_scale(s_tiles.scalar_type()) && s_tiles.dim() == 3 && s_tiles.size(0) == geom::col_blocks(N) &&
                    s_tiles.size(1) == geom::num_groups(K, group) && s_tiles.size(2) == geom::kTileN,
                "w4a8_gemm: s_tiles must be the scale output of w4a8_repack for (N, K, group)");
}

Tensor run_gemm(const Tensor& a_q0, const Tensor& a_scale0, const Tensor& w_tiles, const Tensor& s_tiles, int64_t N,
                int64_t K, int64_t group, bool swiglu) {
    check_geometry("w4a8_gemm", K, group);
    const int64_t kpad = geom::kpad(K, group);
    TORCH_CHECK(a_q0.dim() == 2 && a_q0.scalar_type() == at::kChar, "w4a8_gemm: a_q must be int8 [M, kpad]");
    TORCH_CHECK(a_q0.size(1) == kpad, "w4a8_gemm: a_q has ", a_q0.size(1),
                " columns; the padded group layout of K=", K, ", group=", group, " has ", kpad,
                " (w4a8_quant_pertoken(x, group))");
    TORCH_CHECK(a_scale0.scalar_type() == at::kBFloat16 && a_scale0.dim() == 1 && a_scale0.size(0) == a_q0.size(0),
                "w4a8_gemm: a_scale must be bfloat16 [M]");
    check_weights(w_tiles, s_tiles, N, K, group);
    TORCH_CHECK(!swiglu || N % 32 == 0, "w4a8_gemm_swiglu: N=", N, " must be 2*I with I a multiple of 16");
    const Tensor a_q = rows(a_q0, 16), a_scale = a_scale0.contiguous();
    const int64_t M = a_q.size(0), ncols = swiglu ? N / 2 : N;
    Tensor y = empty({M, ncols}, at::kBFloat16, a_q);
    if (M == 0) return y;
    const Abi& f = abi();
    const int64_t need = f.w4a8_gemm_workspace_bytes(M, N, K, group);
    const Workspace ws = need > 0 ? workspace(a_q, need) : Workspace{};
    check((swiglu ? f.w4a8_gemm_swiglu : f.w4a8_gemm)(a_q.data_ptr(), a_q.stride(0), a_scale.data_ptr(),
                                                      w_tiles.data_ptr(), s_tiles.data_ptr(), scale_code(s_tiles),
                                                      y.data_ptr(), ncols, M, N, K, group, ws.ptr, ws.bytes,
                                                      stream_of(a_q)),
          "w4a8_gemm");
    return y;
}

Tensor gemm(const Tensor& a_q, const Tensor& a_scale, const Tensor& w_tiles, const Tensor& s_tiles, int64_t N,
            int64_t K, int64_t group) {
    return run_gemm(a_q, a_scale, w_tiles, s_tiles, N, K, group, false);
}

Tensor gemm_swiglu(const Tensor& a_q, const Tensor& a_scale, const Tensor& w_tiles, const Tensor& s_tiles, int64_t N,
                   int64_t K, int64_t group) {
    return run_gemm(a_q, a_scale, w_tiles, s_tiles, N, K, group, true);
}

// ------------------------------------------------------------------ quant + GEMM
Tensor linear(const Tensor& x0, const Tensor& w_tiles, const Tensor& s_tiles, int64_t N, int64_t K, int64_t group,
              const std::optional<Tensor>& bias0) {
    TORCH_CHECK(x0.dim() == 2 && x0.scalar_type() == at::kBFloat16, "w4a8_linear: x must be bfloat16 [M, K]");
    TORCH_CHECK(x0.size(1) == K, "w4a8_linear: x has ", x0.size(1), " columns, K=", K);
    check_geometry("w4a8_linear", K, group);
    check_weights(w_tiles, s_tiles, N, K, group);
    std::optional<Tensor> bias;
    if (bias0.has_value()) {
        TORCH_CHECK(bias0->scalar_type() == at::kBFloat16 && bias0->dim() == 1 && bias0->size(0) == N &&
                        bias0->device() == x0.device(),
                    "w4a8_linear: bias must be bfloat16 [N] on the device of x");
        bias = bias0->contiguous();
    }
    const Tensor x = rows(x0);
    const int64_t M = x.size(0), width = geom::kpad(K, group);
    Tensor y = empty({M, N}, at::kBFloat16, x);
    if (M == 0) return y;
    // one scratch tensor: the int8 rows, then the bf16 scales
    const int64_t as_off = (M * width + 255) / 256 * 256;
    const Tensor aq = empty({as_off + 2 * M}, at::kChar, x);
    char* const p = static_cast<char*>(aq.data_ptr());
    const Abi& f = abi();
    // the prefill kernels' epilogue adds the bias; up to kDecodeMaxM rows torch does
    const bool epilogue = bias.has_value() && M > w4a8::kDecodeMaxM;
    const int64_t need = f.w4a8_gemm_workspace_bytes(M, N, K, group);
    const Workspace ws = need > 0 ? workspace(x, need) : Workspace{};
    check(f.w4a8_linear_bias(x.data_ptr(), x.stride(0), w_tiles.data_ptr(), s_tiles.data_ptr(), scale_code(s_tiles),
                             epilogue ? bias->data_ptr() : nullptr, y.data_ptr(), N, p, width, p + as_off, M, N, K,
                             group, ws.ptr, ws.bytes, stream_of(x)),
          "w4a8_linear");
    if (bias.has_value() && !epilogue) {
        at::AutoDispatchBelowADInplaceOrView guard;   // the op has no derivative, with any row count
        y.add_(*bias);
    }
    return y;
}

// ------------------------------------------------------------------ RMSNorm + quant
std::tuple<Tensor, Tensor, Tensor, Tensor> rmsnorm_quant(const Tensor& x0, const Tensor& weight0, double eps,
                                                         const std::optional<Tensor>& residual0, int64_t group,
                                                         bool want_normed) {
    TORCH_CHECK(x0.dim() == 2 && x0.scalar_type() == at::kBFloat16, "w4a8_rmsnorm_quant: x must be bfloat16 [M, K]");
    const int64_t M = x0.size(0), K = x0.size(1);
    TORCH_CHECK(weight0.scalar_type() == at::kBFloat16 && weight0.dim() == 1 && weight0.size(0) == K,
                "w4a8_rmsnorm_quant: weight must be bfloat16 [K]");
    const Tensor x = rows(x0, 8), weight = weight0.contiguous();
    Tensor residual, s;
    if (residual0.has_value()) {
        TORCH_CHECK(residual0->scalar_type() == at::kBFloat16 && residual0->sizes() == x.sizes(),
                    "w4a8_rmsnorm_quant: residual must match x");
        residual = rows(*residual0, 8);
        s = at::empty_like(x);
    } else {
        s = empty({0, K}, at::kBFloat16, x);
    }
    const int64_t width = quant_width(K, group);
    Tensor a_q = empty({M, width}, at::kChar, x), a_scale = empty({M}, at::kBFloat16, x);
    Tensor h = empty({want_normed ? M : 0, K}, at::kBFloat16, x);
    if (M)
        check(abi().w4a8_rmsnorm_quant(x.data_ptr(), x.stride(0), residual.defined() ? residual.data_ptr() : nullptr,
                                       residual.defined() ? residual.stride(0) : 0, weight.data_ptr(),
                                       static_cast<float>(eps), residual.defined() ? s.data_ptr() : nullptr, K,
                                       want_normed ? h.data_ptr() : nullptr, K, a_q.data_ptr(), width,
                                       a_scale.data_ptr(), M, K, group, stream_of(x)),
              "w4a8_rmsnorm_quant");
    return {a_q, a_scale, s, h};
}

// ------------------------------------------------------------------ RoPE + KV-cache append
void check_tables(const char* op, const Tensor& cos, const Tensor& sin, int64_t L, int64_t D) {
    for (const auto& [t, name] : {std::pair<const Tensor&, const char*>{cos, "cos"}, {sin, "sin"}})
        TORCH_CHECK(t.dim() == 2 && t.scalar_type() == at::kFloat && t.size(0) >= L && t.size(1) >= D / 2 &&
                        t.stride(1) == 1,
                    op, ": ", name, " must be float32 [>= L, >= head_dim / 2]");
    TORCH_CHECK(cos.stride(0) == sin.stride(0), op, ": cos and sin must share a row stride");
}

std::optional<Tensor> check_bias(const char* op, const std::optional<Tensor>& bias, int64_t W, const Tensor& qkv) {
    if (!bias.has_value()) return std::nullopt;
    TORCH_CHECK(bias->scalar_type() == at::kBFloat16 && bias->numel() == W && bias->device() == qkv.device(), op,
                ": bias must be bfloat16 [(heads + 2 kv_heads) * head_dim] on the device");
    return bias->contiguous();
}

Tensor rope_kv(const Tensor& qkv0, const Tensor& cos, const Tensor& sin, const Tensor& pos, const Tensor& k_cache,
               const Tensor& v_cache, int64_t heads, int64_t kv_heads, const std::optional<Tensor>& bias0) {
    TORCH_CHECK(qkv0.dim() == 3 && qkv0.scalar_type() == at::kBFloat16, "w4a8_rope_kv: qkv must be bfloat16 [B, T, W]");
    const int64_t B = qkv0.size(0), T = qkv0.size(1), W = qkv0.size(2);
    TORCH_CHECK(heads > 0 && kv_heads > 0 && W % (heads + 2 * kv_heads) == 0,
                "w4a8_rope_kv: qkv width must be (heads + 2 kv_heads) * head_dim");
    const int64_t D = W / (heads + 2 * kv_heads);
    TORCH_CHECK(D % 2 == 0, "w4a8_rope_kv: head_dim must be even");
    TORCH_CHECK(k_cache.dim() == 4 && v_cache.dim() == 4 && k_cache.scalar_type() == at::kBFloat16 &&
                    v_cache.scalar_type() == at::kBFloat16,
                "w4a8_rope_kv: caches must be 4-D bfloat16");
    const int64_t L = k_cache.size(3);
    TORCH_CHECK(k_cache.sizes() == at::IntArrayRef({B, kv_heads, D, L}) &&
                    v_cache.sizes() == at::IntArrayRef({B, kv_heads, L, D}),
                "w4a8_rope_kv: caches must be k [B, kv_heads, D, L] and v [B, kv_heads, L, D]");
    check_tables("w4a8_rope_kv", cos, sin, L, D);
    TORCH_CHECK(pos.scalar_type() == at::kLong && pos.numel() == 1 && pos.device() == qkv0.device(),
                "w4a8_rope_kv: pos must be one int64 on the device (the position of token 0, shared by every "
                "sequence; per-sequence positions are not supported)");
    const Tensor qkv = qkv0.stride(2) != 1 || qkv0.stride(0) != T * qkv0.stride(1) ? qkv0.contiguous() : qkv0;
    const auto bias = check_bias("w4a8_rope_kv", bias0, W, qkv);
    Tensor q = empty({B, T, heads, D}, at::kBFloat16, qkv);
    if (B * T)
        check(abi().w4a8_rope_kv(qkv.data_ptr(), qkv.stride(1), opt_ptr(bias), cos.data_ptr(), sin.data_ptr(),
                                 cos.stride(0), L, pos.data_ptr(), q.data_ptr(), k_cache.data_ptr(),
                                 k_cache.strides().data(), v_cache.data_ptr(), v_cache.strides().data(), B, T, heads,
                                 kv_heads, D, stream_of(qkv)),
              "w4a8_rope_kv");
    return q;
}

// ------------------------------------------------------------------ attention
float softmax_scale(const std::optional<double>& scale, int64_t D) {
    return static_cast<float>(scale.has_value() ? *scale : 1.0 / std::sqrt(static_cast<double>(D)));
}

Tensor attention(const Tensor& q0, const Tensor& k_cache, const Tensor& vt_cache, const Tensor& pos, int64_t L,
                 int64_t cps, bool split, const std::optional<double>& scale) {
    TORCH_CHECK(q0.dim() == 4 && q0.scalar_type() == at::kBFloat16, "w4a8_attention: q must be bfloat16 [B, T, H, D]");
    const int64_t B = q0.size(0), T = q0.size(1), H = q0.size(2), D = q0.size(3);
    TORCH_CHECK(k_cache.dim() == 4 && vt_cache.dim() == 4 && k_cache.scalar_type() == at::kBFloat16 &&
                    vt_cache.scalar_type() == at::kBFloat16,
                "w4a8_attention: caches must be 4-D bfloat16");
    const int64_t KVH = k_cache.size(1), Lc = k_cache.size(2);
    TORCH_CHECK(k_cache.sizes() == at::IntArrayRef({B, KVH, Lc, D}) &&
                    vt_cache.sizes() == at::IntArrayRef({B, KVH, D, Lc}),
                "w4a8_attention: caches must be k [B, kv_heads, Lc, D] and vt [B, kv_heads, D, Lc]");
    TORCH_CHECK(k_cache.is_contiguous() && vt_cache.is_contiguous(), "w4a8_attention: caches must be contiguous");
    TORCH_CHECK(pos.scalar_type() == at::kLong && pos.numel() == 1 && pos.device() == q0.device(),
                "w4a8_attention: pos must be one int64 on the device");
    const Tensor q = q0.contiguous();
    Tensor out = at::empty_like(q);
    if (B * T == 0) return out;
    const Abi& f = abi();
    Workspace ws;
    if (split) {
        const int64_t need = f.w4a8_attention_workspace_bytes(B, T, H, D, Lc, cps);
        TORCH_CHECK(need >= 0, "w4a8_attention: bad shape for the workspace size");
        ws = workspace(q, std::max<int64_t>(need, 16));
    }
    check(f.w4a8_attention(q.data_ptr(), k_cache.data_ptr(), vt_cache.data_ptr(), out.data_ptr(), pos.data_ptr(), B, T,
                           H, KVH, D, L, Lc, cps, softmax_scale(scale, D), ws.ptr, ws.bytes, stream_of(q)),
          "w4a8_attention");
    return out;
}

Tensor attention_rope(const Tensor& qkv0, const Tensor& cos, const Tensor& sin, const Tensor& pos,
                      const Tensor& k_cache, const Tensor& vt_cache, int64_t heads, int64_t kv_heads, int64_t L,
                      int64_t cps, const std::optional<Tensor>& bias0, const std::optional<double>& scale) {
    TORCH_CHECK(qkv0.dim() == 2 && qkv0.scalar_type() == at::kBFloat16,
                "w4a8_attention_rope: qkv must be bfloat16 [B, W]");
    const int64_t B = qkv0.size(0), W = qkv0.size(1);
    TORCH_CHECK(heads > 0 && kv_heads > 0 && W % (heads + 2 * kv_heads) == 0,
                "w4a8_attention_rope: qkv width must be (heads + 2 kv_heads) * head_dim");
    const int64_t D = W / (heads + 2 * kv_heads);
    TORCH_CHECK(k_cache.dim() == 4 && vt_cache.dim() == 4 && k_cache.scalar_type() == at::kBFloat16 &&
                    vt_cache.scalar_type() == at::kBFloat16,
                "w4a8_attention_rope: caches must be 4-D bfloat16");
    const int64_t Lc = k_cache.size(2);
    TORCH_CHECK(k_cache.sizes() == at::IntArrayRef({B, kv_heads, Lc, D}) &&
                    vt_cache.sizes() == at::IntArrayRef({B, kv_heads, D, Lc}) && k_cache.is_contiguous() &&
                    vt_cache.is_contiguous(),
                "w4a8_attention_rope: caches must be contiguous k [B, kv_heads, Lc, D] and vt [B, kv_heads, D, Lc]");
    check_tables("w4a8_attention_rope", cos, sin, L, D);
    TORCH_CHECK(pos.scalar_type() == at::kLong && pos.numel() == 1 && pos.device() == qkv0.device(),
                "w4a8_attention_rope: pos must be one int64 on the device");
    const Tensor qkv = rows(qkv0, 8);
    const auto bias = check_bias("w4a8_attention_rope", bias0, W, qkv);
    Tensor out = empty({B, 1, heads, D}, at::kBFloat16, qkv);
    if (B == 0) return out;
    const Abi& f = abi();
    const int64_t need = f.w4a8_attention_workspace_bytes(B, 1, heads, D, Lc, cps);
    TORCH_CHECK(need >= 0, "w4a8_attention_rope: bad shape for the workspace size");
    const Workspace ws = need > 0 ? workspace(qkv, need) : Workspace{};
    check(f.w4a8_attention_rope(qkv.data_ptr(), qkv.stride(0), opt_ptr(bias), cos.data_ptr(), sin.data_ptr(),
                                cos.stride(0), k_cache.data_ptr(), vt_cache.data_ptr(), out.data_ptr(),
                                pos.data_ptr(), B, heads, kv_heads, D, L, Lc, cps, softmax_scale(scale, D), ws.ptr,
                                ws.bytes, stream_of(qkv)),
          "w4a8_attention_rope");
    return out;
}

// ------------------------------------------------------------------ mid-group compat pair
int64_t padded_rows(int64_t M) {
    const int64_t t = M <= 16 ? 16 : (M <= 64 ? 64 : 128);
    return geom::ceil_to(M, t);
}

std::vector<Tensor> midgroup_quant_a(const Tensor& x0, int64_t group) {
    TORCH_CHECK(x0.dim() == 2, "midgroup_quant_a: x must be [M, K]");
    TORCH_CHECK(x0.scalar_type() == at::kBFloat16, "midgroup_quant_a: x must be bfloat16");
    TORCH_CHECK(group > 0, "midgroup_quant_a: group must be > 0");
    const Tensor x = rows(x0);
    const int64_t M = x.size(0), K = x.size(1);
    check_geometry("midgroup_quant_a", K, group);
    const int64_t G = geom::num_groups(K, group), kb = geom::kpad(K, group) / 2, Mp = M ? padded_rows(M) : 0;
    Tensor a_hi = empty({Mp, kb}, at::kChar, x), a_lo = empty({Mp, kb}, at::kChar, x);
    Tensor a_scale = empty({G, Mp}, at::kBFloat16, x), a_ksum = empty({G, Mp}, at::kInt, x);
    if (Mp)
        check(abi().w4a8_midgroup_quant_a(x.data_ptr(), x.stride(0), a_hi.data_ptr(), a_lo.data_ptr(),
                                          a_scale.data_ptr(), a_ksum.data_ptr(), M, Mp, K, group, stream_of(x)),
              "midgroup_quant_a");
    return {a_hi, a_lo, a_scale, a_ksum};
}

// w_q is [N, kpad/2], or with tiled the midgroup_tile_weights tiles of such a weight.
Tensor run_midgroup(const Tensor& a_hi0, const Tensor& a_lo0, const Tensor& a_scale0, const Tensor& a_ksum0,
                    const Tensor& w_q0, const Tensor& w_scale0, const Tensor& w_ksum, const Tensor& w_zero0, int64_t N,
                    int64_t K, int64_t group, int64_t nrows, bool tiled) {
    check_geometry("midgroup_w4a8_gemm", K, group);
    const Abi& f = abi();
    const int64_t kb = geom::kpad(K, group) / 2, G = geom::num_groups(K, group);
    if (tiled) {
        const int64_t nbytes = f.w4a8_midgroup_tiles_bytes(N, K, group);
        TORCH_CHECK(w_q0.scalar_type() == at::kChar && w_q0.numel() == nbytes && w_q0.is_contiguous(),
                    "midgroup_w4a8_gemm_tiled: w_tiles must be the ", nbytes, " int8 bytes of midgroup_tile_weights");
    }
    TORCH_CHECK(a_hi0.dim() == 2 && a_lo0.dim() == 2 && (tiled || w_q0.dim() == 2),
                "midgroup_w4a8_gemm: a_hi/a_lo [M,K/2] and w_q [N,K/2] must be 2-D");
    TORCH_CHECK(a_hi0.scalar_type() == at::kChar && a_lo0.scalar_type() == at::kChar && w_q0.scalar_type() == at::kChar,
                "midgroup_w4a8_gemm: packed int4 planes must be int8 tensors");
    TORCH_CHECK(a_scale0.scalar_type() == at::kBFloat16 && w_scale0.scalar_type() == at::kBFloat16 &&
                    w_zero0.scalar_type() == at::kBFloat16,
                "midgroup_w4a8_gemm: a_scale/w_scale/w_zero must be bfloat16");
    TORCH_CHECK(a_ksum0.scalar_type() == at::kInt && w_ksum.scalar_type() == at::kInt,
                "midgroup_w4a8_gemm: a_ksum/w_ksum must be int32");
    TORCH_CHECK(a_hi0.size(1) == kb && a_lo0.sizes() == a_hi0.sizes() && (tiled || w_q0.size(1) == kb),
                "midgroup_w4a8_gemm: packed row length must be Kpad/2 = ", kb, " for K=", K,
                " (group-padded layout); got a_hi ", a_hi0.size(1), " w_q ", tiled ? kb : w_q0.size(1));
    int64_t M = a_hi0.size(0);
    if (!tiled) N = w_q0.size(0);
    TORCH_CHECK(a_scale0.dim() == 2 && a_scale0.size(0) == G && a_scale0.size(1) >= M &&
                    a_ksum0.sizes() == a_scale0.sizes(),
                "midgroup_w4a8_gemm: a_scale/a_ksum must be group-major [K/group, M]");
    const int64_t gn[2] = {G, N};
    TORCH_CHECK(w_scale0.sizes() == at::IntArrayRef(gn, 2) && w_zero0.sizes() == at::IntArrayRef(gn, 2) &&
                    w_ksum.sizes() == at::IntArrayRef(gn, 2),
                "midgroup_w4a8_gemm: w_scale/w_zero/w_ksum must be group-major [K/group, N]");
    if (nrows >= 0) {
        // the first rows only (the real rows before quant_a's padding): the padding
        // rows' activation planes are then never read
        TORCH_CHECK(nrows <= M, "midgroup_w4a8_gemm: rows=", nrows, " exceeds the ", M, " activation rows");
        M = nrows;
    }
    const Tensor a_hi = a_hi0.contiguous(), a_lo = a_lo0.contiguous(), w_q = w_q0.contiguous();
    const Tensor a_scale = a_scale0.contiguous(), a_ksum = a_ksum0.contiguous();
    const Tensor w_scale = w_scale0.contiguous(), w_zero = w_zero0.contiguous();
    Tensor y = empty({M, N}, at::kBFloat16, a_hi);
    if (M == 0) return y;
    // w_ksum is validated but not read: the activation bytes are rebuilt exactly from
    // the two planes, so the kernel needs no +8 correction.  Few rows on a long K get a
    // workspace for the int32 group sums of a split K, prefill sizes one for the rebuilt
    // rows, allocated per call as the reference host allocates its GEMM workspace
    // (npu_ops/host/midgroup_w4a8_gemm.cpp:116-118).
    Tensor ws;
    if (const int64_t sums = f.w4a8_midgroup_split_workspace_bytes(M, N, K, group)) {
        ws = empty({sums}, at::kByte, a_hi);
        check(f.w4a8_midgroup_gemm_split(a_hi.data_ptr(), a_lo.data_ptr(), a_scale.data_ptr(), a_ksum.data_ptr(), M,
                                         a_scale.stride(0), w_q.data_ptr(), tiled, w_scale.data_ptr(),
                                         w_zero.data_ptr(), y.data_ptr(), N, N, K, group, ws.data_ptr(), sums,
                                         stream_of(a_hi)),
              "midgroup_w4a8_gemm");
        return y;
    }
    const int64_t need = f.w4a8_midgroup_gemm_workspace_bytes(M, N, K, group);
    if (need) ws = empty({need}, at::kByte, a_hi);
    check((tiled ? f.w4a8_midgroup_gemm_tiled : f.w4a8_midgroup_gemm_ws)(
              a_hi.data_ptr(), a_lo.data_ptr(), a_scale.data_ptr(), a_ksum.data_ptr(), M, a_scale.stride(0),
              w_q.data_ptr(), w_scale.data_ptr(), w_zero.data_ptr(), y.data_ptr(), N, nullptr, N, K, group,
              need ? ws.data_ptr() : nullptr, need, stream_of(a_hi)),
          "midgroup_w4a8_gemm");
    return y;
}

Tensor midgroup_gemm(const Tensor& a_hi, const Tensor& a_lo, const Tensor& a_scale, const Tensor& a_ksum,
                     const Tensor& w_q, const Tensor& w_scale, const Tensor& w_ksum, const Tensor& w_zero, int64_t K,
                     int64_t group, int64_t nrows) {
    return run_midgroup(a_hi, a_lo, a_scale, a_ksum, w_q, w_scale, w_ksum, w_zero, -1, K, group, nrows, false);
}

Tensor midgroup_gemm_tiled(const Tensor& a_hi, const Tensor& a_lo, const Tensor& a_scale, const Tensor& a_ksum,
                           const Tensor& w_tiles, const Tensor& w_scale, const Tensor& w_ksum, const Tensor& w_zero,
                           int64_t N, int64_t K, int64_t group, int64_t nrows) {
    return run_midgroup(a_hi, a_lo, a_scale, a_ksum, w_tiles, w_scale, w_ksum, w_zero, N, K, group, nrows, true);
}

TORCH_LIBRARY_IMPL(npu, CUDA, m) {
    m.impl("w4a8_quant_pertoken", &quant_pertoken);
    m.impl("w4a8_gemm", &gemm);
    m.impl("w4a8_gemm_swiglu", &gemm_swiglu);
    m.impl("w4a8_linear", &linear);
    m.impl("w4a8_rmsnorm_quant", &rmsnorm_quant);
    m.impl("w4a8_rope_kv", &rope_kv);
    m.impl("w4a8_attention", &attention);
    m.impl("w4a8_attention_rope", &attention_rope);
    m.impl("midgroup_quant_a", &midgroup_quant_a);
    m.impl("midgroup_w4a8_gemm", &midgroup_gemm);
    m.impl("midgroup_w4a8_gemm_tiled", &midgroup_gemm_tiled);
}

}  // namespace

PYBIND11_MODULE(w4a8_torch, m) {
    m.def("abi_names", &abi_names);
    m.def("init", [](py::object loader, py::object ws) {
        g_loader = loader.release().ptr();
        g_workspace = ws.release().ptr();
    });
}
