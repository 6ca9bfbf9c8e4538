"""torch.ops.npu.* -- the W4A8 op surface on PyTorch-ROCm.

Keeps the reference's registration namespace ``npu`` (the reference defines
its ops with TORCH_LIBRARY_FRAGMENT(npu, ...), npu_ops/host/midgroup_quant_a.cpp:87-91
and npu_ops/host/midgroup_w4a8_gemm.cpp:149-153) and adds the per-token /
group-size-parameterised ops of this build:

    torch.ops.npu.w4a8_quant_pertoken(x, group=0) -> (a_q, a_scale)
    torch.ops.npu.w4a8_repack(w_q, w_scale, K, group) -> (w_tiles, s_tiles)
    torch.ops.npu.w4a8_gemm(a_q, a_scale, w_tiles, s_tiles, N, K, group) -> y
    torch.ops.npu.w4a8_gemm_partials(a_q, a_scale, w_tiles, s_tiles, N, K, group) -> (y, partials)
    torch.ops.npu.w4a8_gemm_swiglu(a_q, a_scale, w_tiles, s_tiles, N, K, group) -> y [M, N/2]
    torch.ops.npu.w4a8_linear(x, w_tiles, s_tiles, N, K, group, bias=None) -> y   (quant + GEMM, + bf16 [N] bias)

and two producer-side helpers of the decoder forward that drives them:

    torch.ops.npu.w4a8_rmsnorm_quant(x, weight, eps, residual=None, group=0, want_normed=False)
        -> (a_q, a_scale, s, h)
    torch.ops.npu.w4a8_rope_kv(qkv, cos, sin, pos, k_cache, v_cache, heads, kv_heads, bias=None) -> q
    torch.ops.npu.w4a8_attention(q, k_cache, vt_cache, pos, L, chunks_per_split, split=False, scale=None) -> out
    torch.ops.npu.w4a8_attention_rope(qkv, cos, sin, pos, k_cache, vt_cache, heads, kv_heads, L,
                                      chunks_per_split, bias=None, scale=None) -> out   (decode step: rope_kv fused in)

and, with the reference's own names and schemas (group appended with the
reference's fixed value as default), its mid-group compat pair:

    torch.ops.npu.midgroup_quant_a(x, group=1024) -> [a_hi, a_lo, a_scale, a_ksum]
    torch.ops.npu.midgroup_w4a8_gemm(a_hi, a_lo, a_scale, a_ksum, w_q, w_scale, w_ksum, w_zero,
                                     K, group=1024, rows=-1) -> y   (rows >= 0: only the first rows)
    torch.ops.npu.midgroup_w4a8_gemm_partials(...) -> (y, partials)   (parity hook)

and the same GEMM on a weight reordered once at load time (1 KB tiles, the
same bytes; what the compat linear module and vLLM method keep):

    torch.ops.npu.midgroup_tile_weights(w_q, K, group=1024) -> w_tiles
    torch.ops.npu.midgroup_w4a8_gemm_tiled(a_hi, a_lo, a_scale, a_ksum, w_tiles, w_scale, w_ksum, w_zero,
                                           N, K, group=1024, rows=-1) -> y

Only the CUDA (= HIP on ROCm) dispatch key and fake (meta) kernels are
registered: CPU tensors raise, there is no fallback path.  Each impl checks
dtypes and shapes like the reference's host impls (TORCH_CHECK ->
RuntimeError, npu_ops/host/midgroup_w4a8_gemm.cpp:51-85), allocates outputs
with torch, and calls the C ABI on the current stream without synchronising.
The impls of the ops a forward pass calls are in C++ (csrc/torch_ops.cpp, built
into ``_lib/w4a8_torch.so`` and loaded here); the load-time ops and the parity
hooks (repack, tile_weights, the partial dumps) are below in Python.
"""
from __future__ import annotations

import ctypes
import importlib.util
from typing import Dict, Tuple

import torch

from . import _abi
from . import geometry as geo

_LIB = torch.library.Library("npu", "FRAGMENT")
_LIB.define("w4a8_quant_pertoken(Tensor x, int group=0) -> (Tensor, Tensor)")
_LIB.define("w4a8_repack(Tensor w_q, Tensor w_scale, int K, int group) -> (Tensor, Tensor)")
_LIB.define("w4a8_gemm(Tensor a_q, Tensor a_scale, Tensor w_tiles, Tensor s_tiles, "
            "int N, int K, int group) -> Tensor")
_LIB.define("w4a8_gemm_partials(Tensor a_q, Tensor a_scale, Tensor w_tiles, Tensor s_tiles, "
            "int N, int K, int group) -> (Tensor, Tensor)")
_LIB.define("w4a8_gemm_swiglu(Tensor a_q, Tensor a_scale, Tensor w_tiles, Tensor s_tiles, "
            "int N, int K, int group) -> Tensor")
_LIB.define("w4a8_linear(Tensor x, Tensor w_tiles, Tensor s_tiles, int N, int K, int group, Tensor? bias=None) "
            "-> Tensor")
_LIB.define("w4a8_rmsnorm_quant(Tensor x, Tensor weight, float eps, Tensor? residual=None, int group=0, "
            "bool want_normed=False) -> (Tensor, Tensor, Tensor, Tensor)")
_LIB.define("w4a8_rope_kv(Tensor qkv, Tensor cos, Tensor sin, Tensor pos, Tensor(a!) k_cache, Tensor(b!) v_cache, "
            "int heads, int kv_heads, Tensor? bias=None) -> Tensor")
_LIB.define("w4a8_attention(Tensor q, Tensor k_cache, Tensor vt_cache, Tensor pos, int L, int chunks_per_split, "
            "bool split=False, float? scale=None) -> Tensor")
_LIB.define("w4a8_attention_rope(Tensor qkv, Tensor cos, Tensor sin, Tensor pos, Tensor(a!) k_cache, "
            "Tensor(b!) vt_cache, int heads, int kv_heads, int L, int chunks_per_split, Tensor? bias=None, "
            "float? scale=None) -> Tensor")
_LIB.define("midgroup_quant_a(Tensor x, int group=1024) -> Tensor[]")
_LIB.define("midgroup_w4a8_gemm(Tensor a_hi, Tensor a_lo, Tensor a_scale, Tensor a_ksum, Tensor w_q, "
            "Tensor w_scale, Tensor w_ksum, Tensor w_zero, int K, int group=1024, int rows=-1) -> Tensor")
_LIB.define("midgroup_w4a8_gemm_partials(Tensor a_hi, Tensor a_lo, Tensor a_scale, Tensor a_ksum, Tensor w_q, "
            "Tensor w_scale, Tensor w_ksum, Tensor w_zero, int K, int group=1024) -> (Tensor, Tensor)")
_LIB.define("midgroup_tile_weights(Tensor w_q, int K, int group=1024) -> Tensor")
_LIB.define("midgroup_w4a8_gemm_tiled(Tensor a_hi, Tensor a_lo, Tensor a_scale, Tensor a_ksum, Tensor w_tiles, "
            "Tensor w_scale, Tensor w_ksum, Tensor w_zero, int N, int K, int group=1024, int rows=-1) -> Tensor")

_SCALE_DT = {torch.float16: _abi.W4A8_DT_F16, torch.bfloat16: _abi.W4A8_DT_BF16}


def _require(cond: bool, msg: str) -> None:
    if not cond:
        raise RuntimeError(msg)


def _stream(dev: torch.device) -> ctypes.c_void_p:
    return ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)


# One workspace per (device, stream), allocated only when the library asks
# for one (decode shapes that split K over workgroups); it only grows.  Eager
# calls on one stream are stream-ordered, so sharing per stream is safe.
_WORKSPACES: Dict[Tuple[int, int], torch.Tensor] = {}
# Calls captured into a HIP graph get a workspace of that capture instead:
# the graph may be replayed on any stream, while eager calls keep using the
# stream's own, so the two never share memory.  Calls inside one graph run in
# its captured order and share the capture's workspace.
_CAPTURE_WS: Dict[Tuple[int, int], torch.Tensor] = {}
# Workspaces replaced by a larger one stay allocated: a captured HIP graph
# keeps the address it was captured with, so that memory must never return
# to the caching allocator (nor may a capture's own workspace).
_RETIRED: list = []

def _capture_id(stream_handle: int) -> int:
    """The HIP capture sequence id of a stream that is being captured, asked
    through the W4A8 library (bound to the HIP runtime the process loaded)."""
    cid = ctypes.c_ulonglong(0)
    rc = _abi.lib().w4a8_stream_capture_id(ctypes.c_void_p(stream_handle), ctypes.byref(cid))
    if rc != 0:
        raise RuntimeError(f"w4a8: could not read the capture id of stream {stream_handle:#x}: "
                           f"{_abi.lib().w4a8_last_error().decode('utf-8', 'replace')}")
    return int(cid.value)


def _workspace(dev: torch.device, need: int) -> torch.Tensor:
    index = dev.index if dev.index is not None else torch.cuda.current_device()
    stream = torch.cuda.current_stream(dev).cuda_stream
    if torch.cuda.is_current_stream_capturing():
        table, key = _CAPTURE_WS, (index, _capture_id(stream))
    else:
        table, key = _WORKSPACES, (index, stream)
    ws = table.get(key)
    if ws is None or ws.numel() < need:
        if ws is not None:
            _RETIRED.append(ws)
        # no clearing needed: the split GEMM writes every sum the reduce reads
        ws = torch.empty(max(need, 1 << 20), dtype=torch.uint8, device=dev)
        table[key] = ws
    return ws


# ---------------------------------------------------------------- C++ kernels
def _without_native(error: type, why: str) -> None:
    """The native ops raise when called; everything on the host works without them."""
    def missing(*args, **kwargs):
        raise error(f"{why}; build it with `python -c 'import __graft_entry__ as g; g.build()'`")
    for op in ("w4a8_quant_pertoken", "w4a8_gemm", "w4a8_gemm_swiglu", "w4a8_linear", "w4a8_rmsnorm_quant",
               "w4a8_rope_kv", "w4a8_attention", "w4a8_attention_rope", "midgroup_quant_a", "midgroup_w4a8_gemm",
               "midgroup_w4a8_gemm_tiled"):
        _LIB.impl(op, missing, "CUDA")


def _load_native() -> None:
    """Load csrc/torch_ops.cpp's library: importing it registers its ops' CUDA kernels.
    Not built, those ops raise FileNotFoundError when called; not loadable (built for another
    torch, or this torch has no HIP), ImportError."""
    path = _abi.TORCH_LIB_PATH
    if not path.exists():
        _without_native(FileNotFoundError, f"W4A8 torch library not found at {path}")
        return
    try:
        spec = importlib.util.spec_from_file_location("w4a8_torch", str(path))
        native = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(native)
    except ImportError as e:
        _without_native(ImportError, f"W4A8 torch library {path} cannot be loaded ({e})")
        return

    def addresses():
        # the C ABI library, loaded at the first call of an op
        lib = _abi.lib()
        return [ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in native.abi_names()]

    def workspace(index: int, need: int):
        ws = _workspace(torch.device("cuda", index), need)
        return ws.data_ptr(), ws.numel()

    native.init(addresses, workspace)


_load_native()


# ---------------------------------------------------------------- quant
def _quant_width(K: int, group: int) -> int:
    # group > 0: the GEMM's padded group layout (kpad == K when nothing is padded)
    return geo.kpad(K, group) if group > 0 else K


@torch.library.register_fake("npu::w4a8_quant_pertoken")
def _quant_pertoken_fake(x, group=0):
    M, K = x.shape
    return (x.new_empty((M, _quant_width(K, group)), dtype=torch.int8),
            x.new_empty((M,), dtype=torch.bfloat16))


# ---------------------------------------------------------------- repack
def _check_ref_weight(w_q, w_scale, K, group):
    _require(w_q.dim() == 2 and w_q.dtype in (torch.int8, torch.uint8),
             "w4a8_repack: w_q must be a 2-D int8 [N, kpad/2] packed-int4 tensor")
    _require(w_scale.dtype in _SCALE_DT, "w4a8_repack: w_scale must be float16 or bfloat16")
    N = w_q.shape[0]
    G = geo.num_groups(K, group)
    _require(w_q.shape[1] == geo.kpad(K, group) // 2,
             f"w4a8_repack: packed row length must be kpad/2 = {geo.kpad(K, group) // 2} "
             f"for K={K}, group={group}; got {w_q.shape[1]}")
    _require(tuple(w_scale.shape) == (G, N), f"w4a8_repack: w_scale must be group-major [{G}, {N}]")
    return N, G


@torch.library.impl(_LIB, "w4a8_repack", "CUDA")
def _repack_cuda(w_q: torch.Tensor, w_scale: torch.Tensor, K: int, group: int):
    N, G = _check_ref_weight(w_q, w_scale, K, group)
    w_q = w_q.contiguous()
    w_scale = w_scale.contiguous()
    w_tiles = torch.empty((geo.repacked_weight_bytes(N, K, group),), dtype=torch.uint8, device=w_q.device)
    s_tiles = torch.empty(geo.repacked_scale_shape(N, K, group), dtype=w_scale.dtype, device=w_q.device)
    _abi.check(_abi.lib().w4a8_repack(w_q.data_ptr(), w_scale.data_ptr(), _SCALE_DT[w_scale.dtype],
                                      w_tiles.data_ptr(), s_tiles.data_ptr(), N, K, group,
                                      _stream(w_q.device)), "w4a8_repack")
    return w_tiles, s_tiles


@torch.library.register_fake("npu::w4a8_repack")
def _repack_fake(w_q, w_scale, K, group):
    N = w_q.shape[0]
    return (w_q.new_empty((geo.repacked_weight_bytes(N, K, group),), dtype=torch.uint8),
            w_scale.new_empty(geo.repacked_scale_shape(N, K, group)))


# ---------------------------------------------------------------- gemm
def _check_gemm(a_q, a_scale, w_tiles, s_tiles, N, K, group):
    _require(a_q.dim() == 2 and a_q.dtype == torch.int8, "w4a8_gemm: a_q must be int8 [M, kpad]")
    _require(a_q.shape[1] == geo.kpad(K, group),
             f"w4a8_gemm: a_q has {a_q.shape[1]} columns; the padded group layout of K={K}, "
             f"group={group} has {geo.kpad(K, group)} (w4a8_quant_pertoken(x, group))")
    _require(a_scale.dtype == torch.bfloat16 and a_scale.dim() == 1 and a_scale.shape[0] == a_q.shape[0],
             "w4a8_gemm: a_scale must be bfloat16 [M]")
    _require(w_tiles.dtype == torch.uint8 and w_tiles.numel() == geo.repacked_weight_bytes(N, K, group),
             "w4a8_gemm: w_tiles must be the uint8 output of w4a8_repack for (N, K, group)")
    _require(s_tiles.dtype in _SCALE_DT and tuple(s_tiles.shape) == geo.repacked_scale_shape(N, K, group),
             "w4a8_gemm: s_tiles must be the scale output of w4a8_repack for (N, K, group)")


@torch.library.register_fake("npu::w4a8_gemm")
def _gemm_fake(a_q, a_scale, w_tiles, s_tiles, N, K, group):
    return a_q.new_empty((a_q.shape[0], N), dtype=torch.bfloat16)


@torch.library.register_fake("npu::w4a8_gemm_swiglu")
def _gemm_swiglu_fake(a_q, a_scale, w_tiles, s_tiles, N, K, group):
    return a_q.new_empty((a_q.shape[0], N // 2), dtype=torch.bfloat16)


@torch.library.impl(_LIB, "w4a8_gemm_partials", "CUDA")
def _gemm_partials_cuda(a_q, a_scale, w_tiles, s_tiles, N: int, K: int, group: int):
    M, dev = a_q.shape[0], a_q.device
    partials = torch.empty((geo.num_groups(K, group), M, N), dtype=torch.int32, device=dev)
    _check_gemm(a_q, a_scale, w_tiles, s_tiles, N, K, group)
    if a_q.stride(1) != 1 or a_q.stride(0) % 16:
        a_q = a_q.contiguous()
    a_scale = a_scale.contiguous()
    y = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
    if M:
        lib = _abi.lib()
        need = lib.w4a8_gemm_workspace_bytes(M, N, K, group)
        ws = _workspace(dev, need) if need > 0 else None
        ws_ptr, ws_bytes = (ws.data_ptr(), ws.numel()) if ws is not None else (None, 0)
        _abi.check(lib.w4a8_gemm_debug_partials(a_q.data_ptr(), a_q.stride(0), a_scale.data_ptr(), w_tiles.data_ptr(),
                                                s_tiles.data_ptr(), _SCALE_DT[s_tiles.dtype], y.data_ptr(), N,
                                                partials.data_ptr(), M, N, K, group, ws_ptr, ws_bytes, _stream(dev)),
                   "w4a8_gemm")
    return y, partials


@torch.library.register_fake("npu::w4a8_gemm_partials")
def _gemm_partials_fake(a_q, a_scale, w_tiles, s_tiles, N, K, group):
    M = a_q.shape[0]
    return (a_q.new_empty((M, N), dtype=torch.bfloat16),
            a_q.new_empty((geo.num_groups(K, group), M, N), dtype=torch.int32))


# ---------------------------------------------------------------- quant + GEMM
@torch.library.register_fake("npu::w4a8_linear")
def _linear_fake(x, w_tiles, s_tiles, N, K, group, bias=None):
    return x.new_empty((x.shape[0], N), dtype=torch.bfloat16)


@torch.library.register_vmap("npu::w4a8_linear", lib=_LIB)
def _linear_vmap(info, in_dims, x, w_tiles, s_tiles, N, K, group, bias=None):
    """Batched biases are added to one product; any other batched operand runs per element."""
    op = torch.ops.npu.w4a8_linear
    args = (x, w_tiles, s_tiles, N, K, group, bias)
    dims = tuple(in_dims) + (None,) * (len(args) - len(in_dims))
    if all(d is None for d in dims[:-1]):
        return op(*args[:-1]) + bias.movedim(dims[-1], 0)[:, None], 0
    each = [op(*(a if d is None else a.select(d, i) for a, d in zip(args, dims))) for i in range(info.batch_size)]
    return torch.stack(each), 0


# ---------------------------------------------------------------- RMSNorm + quant
@torch.library.register_fake("npu::w4a8_rmsnorm_quant")
def _rmsnorm_quant_fake(x, weight, eps, residual=None, group=0, want_normed=False):
    M, K = x.shape
    return (x.new_empty((M, _quant_width(K, group)), dtype=torch.int8), x.new_empty((M,), dtype=torch.bfloat16),
            x.new_empty((M, K) if residual is not None else (0, K)), x.new_empty((M, K) if want_normed else (0, K)))


# ---------------------------------------------------------------- RoPE + KV-cache append
@torch.library.register_fake("npu::w4a8_rope_kv")
def _rope_kv_fake(qkv, cos, sin, pos, k_cache, v_cache, heads, kv_heads, bias=None):
    B, T, W = qkv.shape
    return qkv.new_empty((B, T, heads, W // (heads + 2 * kv_heads)))


# ---------------------------------------------------------------- attention over the KV cache
def attention_chunks_per_split(batch: int, heads: int, kv_heads: int, cache_len: int) -> int:
    """The split size (in chunks of 64 positions) the library picks for a decode step of
    `batch` sequences over a cache axis of cache_len positions (a multiple of 64)."""
    cps = _abi.lib().w4a8_attention_chunks_per_split(batch, heads, kv_heads, cache_len)
    _require(cps > 0, f"w4a8_attention: bad shape for the split size (B={batch}, H={heads}, KVH={kv_heads}, "
             f"Lc={cache_len})")
    return int(cps)


@torch.library.register_fake("npu::w4a8_attention")
def _attention_fake(q, k_cache, vt_cache, pos, L, chunks_per_split, split=False, scale=None):
    return torch.empty_like(q)


@torch.library.register_fake("npu::w4a8_attention_rope")
def _attention_rope_fake(qkv, cos, sin, pos, k_cache, vt_cache, heads, kv_heads, L, chunks_per_split, bias=None,
                         scale=None):
    B, W = qkv.shape
    return qkv.new_empty((B, 1, heads, W // (heads + 2 * kv_heads)))


# ---------------------------------------------------------------- mid-group compat pair
def tile_m_for(M: int) -> int:
    """Row padding unit of the reference's compat pair (npu_ops/host/midgroup_quant_a.cpp:37)."""
    return 16 if M <= 16 else (64 if M <= 64 else 128)


def _padded_rows(M: int) -> int:
    t = tile_m_for(M)
    return -(-M // t) * t


@torch.library.register_fake("npu::midgroup_quant_a")
def _midgroup_quant_a_fake(x, group=1024):
    M, K = x.shape
    G, kb = geo.num_groups(K, group), geo.kpad(K, group) // 2
    Mp = _padded_rows(M) if M else 0
    return [x.new_empty((Mp, kb), dtype=torch.int8), x.new_empty((Mp, kb), dtype=torch.int8),
            x.new_empty((G, Mp), dtype=torch.bfloat16), x.new_empty((G, Mp), dtype=torch.int32)]


def _check_midgroup(a_hi, a_lo, a_scale, a_ksum, w_q, w_scale, w_ksum, w_zero, K, group):
    # the reference's checks (npu_ops/host/midgroup_w4a8_gemm.cpp:51-85); N % 128 is not required here
    _require(a_hi.dim() == 2 and a_lo.dim() == 2 and w_q.dim() == 2,
             "midgroup_w4a8_gemm: a_hi/a_lo [M,K/2] and w_q [N,K/2] must be 2-D")
    _require(a_hi.dtype == torch.int8 and a_lo.dtype == torch.int8 and w_q.dtype == torch.int8,
             "midgroup_w4a8_gemm: packed int4 planes must be int8 tensors")
    _require(a_scale.dtype == torch.bfloat16 and w_scale.dtype == torch.bfloat16 and w_zero.dtype == torch.bfloat16,
             "midgroup_w4a8_gemm: a_scale/w_scale/w_zero must be bfloat16")
    _require(a_ksum.dtype == torch.int32 and w_ksum.dtype == torch.int32,
             "midgroup_w4a8_gemm: a_ksum/w_ksum must be int32")
    kb = geo.kpad(K, group) // 2
    _require(a_hi.shape[1] == kb and a_lo.shape == a_hi.shape and w_q.shape[1] == kb,
             f"midgroup_w4a8_gemm: packed row length must be Kpad/2 = {kb} for K={K} (group-padded layout); "
             f"got a_hi {a_hi.shape[1]} w_q {w_q.shape[1]}")
    M, N, G = a_hi.shape[0], w_q.shape[0], geo.num_groups(K, group)
    _require(a_scale.dim() == 2 and a_scale.shape[0] == G and a_scale.shape[1] >= M and a_ksum.shape == a_scale.shape,
             "midgroup_w4a8_gemm: a_scale/a_ksum must be group-major [K/group, M]")
    _require(tuple(w_scale.shape) == (G, N) and tuple(w_zero.shape) == (G, N) and tuple(w_ksum.shape) == (G, N),
             "midgroup_w4a8_gemm: w_scale/w_zero/w_ksum must be group-major [K/group, N]")
    return M, N, G


@torch.library.register_fake("npu::midgroup_w4a8_gemm")
def _midgroup_gemm_fake(a_hi, a_lo, a_scale, a_ksum, w_q, w_scale, w_ksum, w_zero, K, group=1024, rows=-1):
    return a_scale.new_empty((a_hi.shape[0] if rows < 0 else rows, w_q.shape[0]), dtype=torch.bfloat16)


@torch.library.impl(_LIB, "midgroup_w4a8_gemm_partials", "CUDA")
def _midgroup_gemm_partials_cuda(a_hi, a_lo, a_scale, a_ksum, w_q, w_scale, w_ksum, w_zero, K: int,
                                 group: int = 1024):
    M, N, G = _check_midgroup(a_hi, a_lo, a_scale, a_ksum, w_q, w_scale, w_ksum, w_zero, K, group)
    a_hi, a_lo, w_q = a_hi.contiguous(), a_lo.contiguous(), w_q.contiguous()
    a_scale, a_ksum = a_scale.contiguous(), a_ksum.contiguous()
    w_scale, w_zero = w_scale.contiguous(), w_zero.contiguous()
    dev = a_hi.device
    y = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
    P = torch.empty((G, M, N), dtype=torch.int32, device=dev)
    if M:
        _abi.check(_abi.lib().w4a8_midgroup_gemm_ws(a_hi.data_ptr(), a_lo.data_ptr(), a_scale.data_ptr(),
                                                    a_ksum.data_ptr(), M, a_scale.stride(0), w_q.data_ptr(),
                                                    w_scale.data_ptr(), w_zero.data_ptr(), y.data_ptr(), N,
                                                    P.data_ptr(), N, K, group, None, 0, _stream(dev)),
                   "midgroup_w4a8_gemm")
    return y, P


@torch.library.impl(_LIB, "midgroup_tile_weights", "CUDA")
def _midgroup_tile_weights_cuda(w_q, K: int, group: int = 1024):
    """w_q [N, kpad/2] -> the 1 KB tiles midgroup_w4a8_gemm_tiled reads (the same bytes)."""
    _require(w_q.dim() == 2 and w_q.dtype == torch.int8, "midgroup_tile_weights: w_q must be int8 [N, kpad/2]")
    _require(w_q.shape[1] == geo.kpad(K, group) // 2,
             f"midgroup_tile_weights: packed row length must be Kpad/2 = {geo.kpad(K, group) // 2} for K={K}")
    w_q = w_q.contiguous()
    N = w_q.shape[0]
    out = torch.empty(max(0, _abi.lib().w4a8_midgroup_tiles_bytes(N, K, group)), dtype=torch.int8, device=w_q.device)
    if N:
        _abi.check(_abi.lib().w4a8_midgroup_tile_weights(w_q.data_ptr(), out.data_ptr(), N, K, group,
                                                         _stream(w_q.device)), "midgroup_tile_weights")
    return out


@torch.library.register_fake("npu::midgroup_tile_weights")
def _midgroup_tile_weights_fake(w_q, K, group=1024):
    N, KT = w_q.shape[0], -(-geo.kpad(K, group) // 128)
    return w_q.new_empty(((N + 15) // 16 * KT * 1024,), dtype=torch.int8)


@torch.library.register_fake("npu::midgroup_w4a8_gemm_tiled")
def _midgroup_gemm_tiled_fake(a_hi, a_lo, a_scale, a_ksum, w_tiles, w_scale, w_ksum, w_zero, N, K, group=1024,
                              rows=-1):
    return a_scale.new_empty((a_hi.shape[0] if rows < 0 else rows, N), dtype=torch.bfloat16)


@torch.library.register_fake("npu::midgroup_w4a8_gemm_partials")
def _midgroup_gemm_partials_fake(a_hi, a_lo, a_scale, a_ksum, w_q, w_scale, w_ksum, w_zero, K, group=1024):
    M, N, G = a_hi.shape[0], w_q.shape[0], geo.num_groups(K, group)
    return (a_scale.new_empty((M, N), dtype=torch.bfloat16), a_scale.new_empty((G, M, N), dtype=torch.int32))
