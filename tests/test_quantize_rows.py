"""quantize_rows: the kernel (hipgemm_quantize_rows_e4m3) against the tensor
operations it stands for, bit for bit, and the calls that keep those
operations.  (That they in turn round to e4m3 correctly is
test_torch_ops.py's part.)"""
import pytest
import torch

import hipgemm_amd as hg
import hipgemm_amd.torch_ops as ops
from util import say

FAKE = 1 << 20


def test_argument_validation():
    L = hg.lib()

    def call(x=FAKE, type=1, M=4, K=64, ldx=64, q=FAKE, s=FAKE):
        return L.hipgemm_quantize_rows_e4m3(x, type, M, K, ldx, q, s, None)
    for kw in (dict(x=None), dict(q=None), dict(s=None), dict(type=3), dict(type=-1),
               dict(M=-1), dict(K=-1), dict(ldx=63), dict(x=FAKE + 1), dict(s=FAKE + 2),
               dict(type=0, x=FAKE + 2)):
        assert call(**kw) == hg.hipErrorInvalidValue, kw
    assert call(M=0, x=None) == 0 and call(K=0, x=None) == 0


def test_cpu_tensors_and_traces_keep_the_tensor_operations(monkeypatch):
    monkeypatch.setattr(ops, "lib", lambda: pytest.fail("kernel path taken"))
    x = torch.randn(5, 48)
    q, s = ops.quantize_rows(x)
    rq, rs = ops._quantize_rows_ops(x)
    assert torch.equal(q.view(torch.uint8), rq.view(torch.uint8)) and torch.equal(s, rs)


def check(x, what):
    say(f"case quantize {what} {tuple(x.shape)} {x.dtype} strides={x.stride()}")
    q, s = ops.quantize_rows(x)
    rq, rs = ops._quantize_rows_ops(x)
    torch.cuda.synchronize()
    assert q.shape == rq.shape and q.dtype == rq.dtype and q.is_contiguous()
    assert torch.equal(s.view(torch.int32), rs.view(torch.int32)), what
    bad = int((q.view(torch.uint8) != rq.view(torch.uint8)).sum())
    assert bad == 0, f"{what}: {bad} of {q.numel()} bytes differ"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [
    (1, 1), (1, 8), (3, 7), (5, 48), (33, 1000),  # less than a load to a few
    (2, 2048), (2, 2056), (4, 8192),              # whole loads per thread
    (2, 16384), (2, 16392),                       # what a 16-bit row keeps
    (2, 8200), (2, 40000), (300, 4099),           # read again; odd
])
def test_kernel_equals_tensor_operations(gpu, dtype, shape):
    g = gpu.Generator(device="cuda").manual_seed(3)
    x = gpu.randn(shape, generator=g, device="cuda")
    x = x * gpu.logspace(-3, 3, shape[0], device="cuda")[:, None]
    check(x.to(dtype), "normal")
    big = gpu.randn((shape[0], shape[1] + 9), generator=g, device="cuda").to(dtype)
    check(big[:, 1:shape[1] + 1], "strided, unaligned rows")


def entry(torch, x):
    """q, s of hipgemm_quantize_rows_e4m3 itself."""
    M, K = x.shape
    q = torch.full((M, K), 0x55, dtype=torch.uint8, device="cuda")
    s = torch.full((M,), -1.0, device="cuda")
    assert hg.lib().hipgemm_quantize_rows_e4m3(
        x.data_ptr(), ops._QUANT_TYPES[x.dtype], M, K, x.stride(0), q.data_ptr(),
        s.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    return q, s


@pytest.mark.gpu
@pytest.mark.parametrize("K", [3, 8])
def test_more_rows_than_one_launch_has_workgroups(gpu, K):
    """2^24 rows and a few: a workgroup per row would be a launch of 2^32
    threads."""
    M = 2 ** 24 + 3
    say(f"case quantize M={M} K={K} bf16")
    g = gpu.Generator(device="cuda").manual_seed(5)
    x = gpu.randn((M, K), generator=g, device="cuda", dtype=gpu.bfloat16)
    q, s = entry(gpu, x)
    rq, rs = ops._quantize_rows_ops(x)
    assert gpu.equal(s, rs) and gpu.equal(q, rq.view(gpu.uint8))


# (M, K, wide loads) -> whether the kernel takes it, for 2-byte elements.
ROUTES = {(16384, 16, True): True, (16392, 16, True): False, (65536, 255, False): True,
          (70000, 248, True): False, (70000, 256, True): True,
          (65536, 3, False): True, (65544, 64, False): False, (65544, 65, False): True,
          (1, 131072, True): True, (255, 131080, True): False, (256, 131080, True): True,
          (1, 20481, False): False, (1023, 20481, False): False,
          (1024, 20481, False): True, (1, 20480, False): True, (1, 256, False): True}


def test_rows_the_kernel_takes():
    """The choice by sizes, for 2- and 4-byte elements, and by alignment."""
    for (M, K, wide), want in ROUTES.items():
        assert ops._kernel_ahead(M, K, K, 2, 4096 if wide else 4098) is want, (M, K, wide)
    assert ops._kernel_ahead(32768, 4, 4, 4, 4096)
    assert not ops._kernel_ahead(32769, 124, 124, 4, 4096)
    assert ops._kernel_ahead(32769, 128, 128, 4, 4096)
    assert ops._kernel_ahead(1, 65536, 65536, 4, 4096)
    assert not ops._kernel_ahead(1, 65540, 65540, 4, 4096)
    assert not ops._kernel_ahead(1, 65536, 65537, 4, 4096)  # stride


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [s for s in ROUTES if s[0] * s[1] < 2 ** 25],
                         ids=lambda s: "x".join(map(str, s)))
def test_kernel_where_it_is_ahead(gpu, monkeypatch, shape):
    """Rows that the kernel is slower on are tensor operations, and the kernel's
    results on them are theirs."""
    M, K, wide = shape
    say(f"case quantize route {M}x{K} wide={wide}")
    x = gpu.randn((M, K + 8), device="cuda", dtype=gpu.bfloat16)
    x = x[:, :K] if wide else x[:, 1:K + 1]
    assert ((x.data_ptr() | 2 * x.stride(0) | 2 * K) % 16 == 0) == wide
    q, s = entry(gpu, x)
    rq, rs = ops._quantize_rows_ops(x)
    assert gpu.equal(s, rs) and gpu.equal(q, rq.view(gpu.uint8))
    calls = []
    real = ops.lib
    monkeypatch.setattr(ops, "lib", lambda: calls.append(1) or real())
    ops.quantize_rows(x)
    assert bool(calls) == ROUTES[shape]


@pytest.mark.gpu
def test_row_of_almost_2_31_elements(gpu):
    """One row of 2^31 - 5 elements, read one by one: the index of a thread's
    next element passes 2^31."""
    K = 2 ** 31 - 5
    say(f"case quantize M=1 K={K} bf16")
    x = gpu.zeros((1, K), dtype=gpu.bfloat16, device="cuda")
    at = gpu.tensor([0, 300, 2 ** 30, K - 300, K - 2, K - 1], device="cuda")
    x[0, at] = gpu.tensor([1.0, -2, 3, -448, 28, 7], device="cuda", dtype=gpu.bfloat16)
    q, s = entry(gpu, x)
    gpu.cuda.synchronize()
    assert s.item() == 1.0
    want = gpu.tensor([1.0, -2, 3, -448, 28, 7], device="cuda").to(gpu.float8_e4m3fn)
    assert gpu.equal(q[0, at], want.view(gpu.uint8))
    assert int(gpu.count_nonzero(q)) == at.numel()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_special_rows(gpu, dtype):
    inf, nan = float("inf"), float("nan")
    f = gpu.finfo(dtype)
    rows = [[0.0] * 8, [-0.0, 0.0] * 4, [inf, 1, -1, 0, 2, 3, 4, 5], [-inf] + [1.0] * 7,
            [nan, 1, 500, -500, 0, -0.0, 448, 449], [nan, inf, -inf, 1, 2, 3, 4, 5],
            [f.tiny, -f.tiny, f.tiny / 2, 0, f.smallest_normal, 0, 0, 0],
            [1e-45, 0, 0, 0, 0, 0, 0, 0], [1e-42, -1e-44, 0, 0, 0, 0, 0, 0],
            [f.max, -f.max, 1, 0, f.max / 2, 3, 4, 5],
            [448, 447, 440, 432, 1, 0.5, 0.0156, 0.001], [1, 2, 4, 8, 16, 32, 64, 128]]
    x = gpu.tensor(rows, device="cuda", dtype=gpu.float64).to(dtype)
    check(x, "special")
    check(gpu.cat([x, x], 1)[:, 3:11], "special, unaligned")


@pytest.mark.gpu
def test_quotients_near_rounding_boundaries(gpu):
    """Rows whose scale has every kind of significand (powers of two, all
    ones, one ulp off) and whose elements lie on, and one ulp to each side of,
    the midpoints between e4m3 values times that scale."""
    import numpy as np
    mids = []
    for e in range(-10, 9):
        for m in range(16):
            mids.append((1 + (2 * m + 1) / 32 if m < 8 else 1 + (m - 8) / 16) * 2.0 ** e)
    base = np.array(mids, np.float64)
    rows = []
    rng = np.random.default_rng(4)
    scales = [1.0, 1.5, 2.0 ** -20, 2.0 ** 30, np.float32(2) - np.float32(2 ** -23),
              np.float32(1) + np.float32(2 ** -23), 1e-30, 3e-38, 2.0 ** -80, 2.0 ** -79]
    scales += list(np.exp2(rng.uniform(-60, 60, 54)))
    for s in scales:
        x = (base * s).astype(np.float32)
        x = np.concatenate([x, np.nextafter(x, np.float32(0)),
                            np.nextafter(x, np.float32(np.inf)), [np.float32(448 * s)]])
        rows.append(np.where(rng.integers(0, 2, x.size) > 0, x, -x).astype(np.float32))
    x = gpu.from_numpy(np.stack(rows)).cuda()
    pad = -x.shape[1] % 8
    check(gpu.nn.functional.pad(x, (0, pad)), "boundaries")


@pytest.mark.gpu
def test_watched_calls_keep_the_tensor_operations(gpu, monkeypatch):
    """Autograd (reverse and forward), vmap, tracing, dispatch modes and other
    layouts see the operations they saw before."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    x = gpu.randn(6, 64, device="cuda")
    want = ops.quantize_rows(x)
    monkeypatch.setattr(ops, "lib", lambda: pytest.fail("kernel path taken"))
    say("case quantize watched calls 6x64")

    def same(got):
        assert gpu.equal(got[0].view(gpu.uint8), want[0].view(gpu.uint8))
        assert gpu.equal(got[1], want[1])
    r = x.clone().requires_grad_()
    q, s = ops.quantize_rows(r)
    s.sum().backward()
    assert r.grad is not None and r.grad.abs().sum() > 0
    same((q.detach(), s.detach()))
    with gpu.autograd.forward_ad.dual_level():
        d = gpu.autograd.forward_ad.make_dual(x, gpu.ones_like(x))
        _, s = ops.quantize_rows(d)
        assert gpu.autograd.forward_ad.unpack_dual(s).tangent is not None
    sv = gpu.func.vmap(lambda t: ops.quantize_rows(t)[1])(x.view(2, 3, 64))
    assert gpu.equal(sv.reshape(-1), want[1])
    gm = make_fx(lambda t: ops.quantize_rows(t)[1])(x)
    assert any("amax" in str(n.target) for n in gm.graph.nodes)
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        q, s = ops.quantize_rows(mode.from_tensor(x))
        assert q.dtype == gpu.float8_e4m3fn and tuple(s.shape) == (6,)
    t = x.t().contiguous().t()  # columns contiguous
    q, s = ops.quantize_rows(t)
    assert gpu.equal(s, want[1])
    with gpu.no_grad():
        monkeypatch.undo()
        same(ops.quantize_rows(r))


@pytest.mark.gpu
def test_layer_equals_operator_path(gpu, monkeypatch):
    """Fp8Linear's direct call against the operator it takes when something
    watches the operations: the same bits, for 2-D, 3-D and empty inputs."""
    gpu.manual_seed(9)
    layer = ops.Fp8Linear.from_linear(gpu.nn.Linear(256, 384).cuda(), activation="silu")
    for shape in ((40, 256), (2, 3, 256), (0, 256), (1, 256)):
        say(f"case fp8-linear direct x={shape}")
        x = gpu.randn(shape, device="cuda", dtype=gpu.bfloat16)
        got = layer(x)
        with monkeypatch.context() as m:
            m.setattr(ops, "_plain_eager", lambda t: False)
            want = layer(x)
        gpu.cuda.synchronize()
        assert got.shape == want.shape == (*shape[:-1], 384)
        assert gpu.equal(got.view(gpu.int16), want.view(gpu.int16))
    x = gpu.randn(4, 256, device="cuda", requires_grad=True)
    assert layer(x).requires_grad
    with gpu.no_grad():
        assert not layer(x).requires_grad
