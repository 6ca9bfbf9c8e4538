"""The C++ torch kernels (csrc/torch_ops.cpp): what is registered, the inputs they
accept and refuse, and calls from several threads."""
from __future__ import annotations

import subprocess
import sys
import threading

import pytest
import torch

from conftest import ROOT

OPS = ["w4a8_quant_pertoken", "w4a8_gemm", "w4a8_gemm_swiglu", "w4a8_linear", "w4a8_rmsnorm_quant", "w4a8_rope_kv",
       "w4a8_attention", "w4a8_attention_rope", "midgroup_quant_a", "midgroup_w4a8_gemm", "midgroup_w4a8_gemm_tiled"]


def test_native_ops_are_registered(pkg):
    assert pkg._abi.TORCH_LIB_PATH.exists(), "csrc/torch_ops.cpp is not built"
    for op in OPS:
        assert torch._C._dispatch_has_kernel_for_dispatch_key(f"npu::{op}", "CUDA"), op
        assert not torch._C._dispatch_has_kernel_for_dispatch_key(f"npu::{op}", "CPU"), op


@pytest.mark.parametrize("content", [None, b"not a library"])
def test_host_side_without_the_native_ops(tmp_path, content):
    """Without the ops' library, or with one this torch cannot load, the package imports, packs
    weights on the CPU and keeps a CUDA kernel per op (one that raises)."""
    lib = tmp_path / "w4a8_torch.so"
    if content is not None:
        lib.write_bytes(content)
    code = f"""
import importlib, importlib.util, pathlib, sys
import torch
import __graft_entry__ as g
spec = importlib.util.spec_from_file_location(g.PKG_NAME, g.PKG_DIR / "__init__.py",
                                              submodule_search_locations=[str(g.PKG_DIR)])
pkg = importlib.util.module_from_spec(spec)
sys.modules[g.PKG_NAME] = pkg
importlib.import_module(g.PKG_NAME + "._abi").TORCH_LIB_PATH = pathlib.Path({str(lib)!r})
spec.loader.exec_module(pkg)
w_q, scale = pkg.packing.quantize_weight(torch.randn(32, 128), 64, torch.bfloat16)
assert w_q.shape == (32, 64) and scale.shape == (2, 32)
for op in {OPS!r}:
    assert torch._C._dispatch_has_kernel_for_dispatch_key("npu::" + op, "CUDA"), op
print("imported")
"""
    res = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert res.returncode == 0 and "imported" in res.stdout, res.stderr


def _weight(dev, N, K, G, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    w_q = torch.randint(-128, 128, (N, K // 2), dtype=torch.int8, device=dev, generator=g)
    ws = (torch.rand((K // G, N), device=dev, generator=g) * 0.018 + 0.002).to(torch.bfloat16)
    return torch.ops.npu.w4a8_repack(w_q, ws, K, G)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 5, 70])
def test_strided_inputs(pkg, dev, M):
    """Row-strided, column-strided and 3-D inputs give the contiguous input's bits."""
    N, K, G = 256, 1024, 128
    w, s = _weight(dev, N, K, G, 3)
    wide = torch.randn((M, 2 * K), device=dev).to(torch.bfloat16)
    x = wide[:, :K].contiguous()
    want = torch.ops.npu.w4a8_linear(x, w, s, N, K, G)
    assert torch.equal(torch.ops.npu.w4a8_linear(wide[:, :K], w, s, N, K, G), want)
    assert torch.equal(torch.ops.npu.w4a8_linear(x.t().contiguous().t(), w, s, N, K, G), want)
    a_q, a_s = torch.ops.npu.w4a8_quant_pertoken(x)
    wide_q = torch.zeros((M, K + 16), dtype=torch.int8, device=dev)
    wide_q[:, :K] = a_q
    odd_q = torch.zeros((M, K + 3), dtype=torch.int8, device=dev)   # rows not a multiple of 16 bytes apart
    odd_q[:, :K] = a_q
    # (a single row counts as contiguous whatever its stride, so its odd stride is refused)
    for q in (a_q, wide_q[:, :K]) + ((odd_q[:, :K],) if M > 1 else ()):
        assert torch.equal(torch.ops.npu.w4a8_gemm(q, a_s, w, s, N, K, G), want)
    assert torch.equal(pkg.linear(x.view(1, M, K), w, s, N, G), want.view(1, M, N))
    assert torch.equal(pkg.linear(x.float(), w, s, N, G), want)
    assert torch.ops.npu.w4a8_linear(x[:0], w, s, N, K, G).shape == (0, N)


def _row_views(row):
    """One row [1, K] under the row strides torch counts as contiguous: K, 1, 0 and an odd one."""
    K = row.numel()
    wide = torch.zeros((2, K + 3), dtype=row.dtype, device=row.device)
    wide[0, :K] = row
    views = {"K": row.reshape(1, K), "1": row.reshape(K, 1).t(), "0": row.reshape(K).expand(4, K)[:1],
             "odd": wide[:1, :K]}
    assert [v.stride(0) for v in views.values()] == [K, 1, 0, K + 3]
    assert all(v.is_contiguous() for v in views.values())
    return views


def test_rows_pass_through_by_their_strides(pkg):
    """Only contiguous rows K apart pass through; every other view comes out that way."""
    x = torch.randn((3, 64)).to(torch.bfloat16)
    rows = pkg.linear.__globals__["_rows"]
    assert rows(x, 64) is x
    cases = list(_row_views(x[0]).values()) + [x.t().contiguous().t(), x.float(), x.view(1, 3, 64), x[:, :32], x[:0]]
    for v in cases:
        got = rows(v, v.shape[-1])
        assert got.dtype is torch.bfloat16 and got.stride() == (v.shape[-1], 1) and got.is_contiguous()
        assert torch.equal(got, v.reshape(-1, v.shape[-1]).to(torch.bfloat16))


@pytest.mark.gpu
def test_one_row_strides(pkg, dev):
    """A single token under every row stride torch counts as contiguous, through each caller."""
    N, K, G = 256, 1024, 128
    w, s = _weight(dev, N, K, G, 3)
    lin = torch.nn.Linear(K, N, bias=True, device=dev)
    modules = [pkg.W4A8Linear.from_float(lin, G), pkg.MidGroupW4A8Linear.from_float(lin, 512)]
    mid = modules[1]
    calls = [lambda x: pkg.linear(x, w, s, N, G), lambda x: pkg.linear_swiglu(x, w, s, N, G), *modules,
             lambda x: pkg.midgroup_linear(x, mid.weight_packed, *mid._gn, 512)]
    views = _row_views(torch.randn((1, K), device=dev).to(torch.bfloat16))
    for i, call in enumerate(calls):
        want = call(views["K"])
        for name, v in views.items():
            assert torch.equal(call(v), want), (i, name)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,G", [
    (1, 5120, 1024, 128),      # fused single row, staged decode plans
    (5, 1000, 1024, 128),      # N off the 16-column tile
    (16, 256, 1024, 64),
    (40, 1000, 2048, 256),     # row groups
    (12, 32800, 256, 128),     # wide kernel
    (20, 1000, 16384, 128),    # wide kernel, K split: added by the reduce
    (50, 1000, 16384, 128),    # split prefill tile
    (12, 512, 16384, 16384),   # one group, int32 sums in the reduce
    (70, 1000, 512, 128),      # 64-row prefill tiles, a ragged last column tile
    (600, 7000, 256, 128),     # 128-row prefill tiles
    (130, 1000, 1024, 64),     # 64 x 64 wave tiles
])
def test_linear_bias(pkg, dev, M, N, K, G):
    """The bias on every plan (past 64 rows in the epilogue): the bits of the bf16 add after the linear."""
    w, s = _weight(dev, N, K, G, M + N)
    x = torch.randn((M, K), device=dev).to(torch.bfloat16)
    bias = torch.randn((N,), device=dev).to(torch.bfloat16)
    y = torch.ops.npu.w4a8_linear(x, w, s, N, K, G)
    assert torch.equal(torch.ops.npu.w4a8_linear(x, w, s, N, K, G, bias), y + bias)
    assert torch.equal(pkg.linear(x, w, s, N, G, bias), y + bias)


@pytest.mark.gpu
def test_linear_bias_left_to_torch(pkg, dev):
    """Biases the epilogue does not take keep torch's own add: dtype promotion,
    broadcasting, autograd and forward-mode derivatives."""
    M, N, K, G = 3, 256, 512, 128
    w, s = _weight(dev, N, K, G, 9)
    x = torch.randn((M, K), device=dev).to(torch.bfloat16)
    y = torch.ops.npu.w4a8_linear(x, w, s, N, K, G)
    f32 = torch.randn((N,), device=dev)
    assert pkg.linear(x, w, s, N, G, f32).dtype == torch.float32
    col = torch.randn((M, 1), device=dev).to(torch.bfloat16)
    assert torch.equal(pkg.linear(x, w, s, N, G, col), y + col)
    b = f32.to(torch.bfloat16).requires_grad_()
    pkg.linear(x, w, s, N, G, b).sum().backward()
    assert b.grad is not None
    with torch.no_grad():
        assert torch.equal(pkg.linear(x, w, s, N, G, b), y + b)
    import torch.autograd.forward_ad as fwd
    with fwd.dual_level():
        dual = fwd.make_dual(b.detach(), torch.ones_like(b))
        assert torch.equal(fwd.unpack_dual(pkg.linear(x, w, s, N, G, dual)).tangent, torch.ones_like(y))
    b2 = torch.stack([b.detach(), -b.detach()])
    assert torch.equal(torch.func.vmap(lambda t: pkg.linear(x, w, s, N, G, t))(b2), y + b2[:, None])
    assert torch.equal(torch.func.grad(lambda t: pkg.linear(x, w, s, N, G, t).sum())(b.detach()),
                       torch.full_like(f32, M, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError):
        torch.ops.npu.w4a8_linear(x, w, s, N, K, G, f32)
    # read by the epilogue: a strided view, an odd offset, infinities and NaN
    special = f32.to(torch.bfloat16)
    special[:3] = torch.tensor([float("inf"), float("-inf"), float("nan")])
    for v in (torch.stack([special, special], 1)[:, 1], torch.cat([special[:1], special])[1:]):
        torch.testing.assert_close(torch.ops.npu.w4a8_linear(x, w, s, N, K, G, v), y + v, rtol=0, atol=0, equal_nan=True)


def test_which_biases_the_op_adds(pkg):
    """Plain bf16 [N] tensors; none that autograd, forward mode or a function transform has to
    see."""
    import torch.autograd.forward_ad as fwd
    takes = pkg.linear.__globals__["_epilogue_bias"]
    x, b = torch.zeros((2, 8), dtype=torch.bfloat16), torch.zeros((4,), dtype=torch.bfloat16)
    seen = []

    def record(t):
        seen.append(takes(t, x, 4))
        return (t * 1).sum()

    assert takes(b, x, 4) and takes(torch.nn.Parameter(b, requires_grad=False), x, 4)
    assert not takes(b.float(), x, 4) and not takes(b[:1], x, 4) and not takes(b.view(1, 4), x, 4)
    trained = b.clone().requires_grad_()
    assert not takes(trained, x, 4)
    with torch.no_grad():
        assert takes(trained, x, 4)
    with fwd.dual_level():
        assert not takes(fwd.make_dual(b, b), x, 4)
    torch.func.vmap(record)(torch.stack([b, b]))
    torch.func.vmap(torch.func.grad(record))(torch.stack([b, b]))
    torch.func.grad(record)(b)
    torch.func.jvp(record, (b,), (b,))
    assert seen == [False] * 4


def test_vmap_over_the_linear(pkg):
    """Biases are batched on one product (nested too); other operands run one by one.  The op's
    kernel stands in as a float product here."""
    calls = []

    def product(x, w_tiles, s_tiles, N, K, group, bias=None):
        calls.append(tuple(x.shape))
        y = (x.float() @ w_tiles.float()).to(torch.bfloat16)
        return y if bias is None else y + bias

    g = torch.Generator().manual_seed(1)
    x = torch.randn((3, 8), generator=g).to(torch.bfloat16)
    w = torch.randn((2, 8, 4), generator=g).to(torch.bfloat16)
    b = torch.randn((5, 2, 4), generator=g).to(torch.bfloat16)
    s = torch.zeros(1)
    with torch.library._scoped_library("npu", "IMPL") as lib:
        lib.impl("w4a8_linear", product, "CPU")

        def f(x, w, b):
            return pkg.linear(x, w, s, 4, 128, b)

        each = torch.stack([f(x, w[0], t) for t in b[:, 0]])
        calls.clear()
        assert torch.equal(torch.func.vmap(lambda t: f(x, w[0], t))(b[:, 0]), each)
        assert torch.equal(torch.func.vmap(lambda t: f(x, w[0], t), in_dims=1)(b[:, 0].t().contiguous()), each)
        nested = torch.func.vmap(torch.func.vmap(lambda t: f(x, w[0], t)))(b)
        assert torch.equal(nested[:, 0], each)
        assert calls == [(3, 8)] * 3
        op = torch.ops.npu.w4a8_linear            # the op's own rule, as traced calls take it
        assert torch.equal(torch.func.vmap(lambda t: op(x, w[0], s, 4, 8, 128, t))(b[:, 0]), each)
        assert calls == [(3, 8)] * 4
        got = torch.func.vmap(f, in_dims=(None, 0, 0))(x, w, b[0])
        assert torch.equal(got, torch.stack([f(x, w[i], b[0, i]) for i in range(2)]))
        got = torch.func.vmap(lambda x: f(x, w[0], None))(torch.stack([x, -x]))
        assert torch.equal(got, torch.stack([f(x, w[0], None), f(-x, w[0], None)]))


@pytest.mark.parametrize("bias", [False, True])
def test_linear_traces_into_one_graph(pkg, bias):
    """torch.compile takes the whole linear, bias included, as one op call."""
    x = torch.randn((70, 256)).to(torch.bfloat16)
    w, s = torch.zeros((4 * 2 * 1024,), dtype=torch.uint8), torch.zeros((4, 2, 16), dtype=torch.bfloat16)
    b = torch.zeros((64,), dtype=torch.bfloat16) if bias else None
    graphs = []

    def backend(gm, example_inputs):
        graphs.append([str(n.target) for n in gm.graph.nodes if n.op == "call_function"])
        return gm.forward

    torch._dynamo.reset()
    fn = torch.compile(lambda x: pkg.linear(x, w, s, 64, 128, b), fullgraph=True, backend=backend)
    with pytest.raises(NotImplementedError):     # traced, then run on the CPU, where the op has no kernel
        fn(x)
    assert graphs == [["npu.w4a8_linear"]]


@pytest.mark.gpu
def test_bad_inputs_raise(pkg, dev):
    N, K, G = 256, 1024, 128
    w, s = _weight(dev, N, K, G, 4)
    x = torch.randn((2, K), device=dev).to(torch.bfloat16)
    for bad in (lambda: torch.ops.npu.w4a8_linear(x.float(), w, s, N, K, G),
                lambda: torch.ops.npu.w4a8_linear(x[:, :512], w, s, N, K, G),
                lambda: torch.ops.npu.w4a8_linear(x, w[:-1], s, N, K, G),
                lambda: torch.ops.npu.w4a8_linear(x, w, s.float(), N, K, G),
                lambda: torch.ops.npu.w4a8_linear(x, w, s, N, K, 0),
                lambda: torch.ops.npu.w4a8_linear(x, w, s, -N, K, G),
                lambda: torch.ops.npu.w4a8_quant_pertoken(x[0]),
                lambda: torch.ops.npu.w4a8_quant_pertoken(x, -1),
                lambda: torch.ops.npu.midgroup_quant_a(x, 0)):
        with pytest.raises(RuntimeError):
            bad()


@pytest.mark.gpu
def test_threads_with_their_own_streams(pkg, dev):
    """Four threads, a stream each, calling a linear whose GEMM splits K (workspace per
    stream) and one whose does not: every result is the single-threaded one."""
    shapes = [(24, 1000 // 16 * 16, 16384, 128), (3, 512, 1024, 128)]
    work = []
    for i, (M, N, K, G) in enumerate(shapes):
        w, s = _weight(dev, N, K, G, 10 + i)
        x = torch.randn((M, K), device=dev).to(torch.bfloat16)
        work.append((x, w, s, N, K, G, torch.ops.npu.w4a8_linear(x, w, s, N, K, G)))
    torch.cuda.synchronize()
    bad = []

    def run(t):
        with torch.cuda.stream(torch.cuda.Stream(device=dev)):
            for i in range(20):
                x, w, s, N, K, G, want = work[(i + t) % len(work)]
                y = torch.ops.npu.w4a8_linear(x, w, s, N, K, G)
                if not torch.equal(y, want):
                    bad.append((t, i))

    ts = [threading.Thread(target=run, args=(t,)) for t in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
