"""GPU parity of AUTO in the regions that the rules of hipgemm_select_variant
name one by one: up to 64 rows (column strips of 32 or 64 columns, one or more
K-slices; 128 x 128 tiles for N > 64 x CUs from 17 rows and, above 48 rows, for
K > 8192), 65-128 rows (strips for a B_T of at most 8 MiB, the split-K schedule on
half-filled K-splits of 3 slices or more, else 128 x 128 tiles), and M > 128
where 128 x 128 tiles take under two rounds while 256 x 256 ones fill at most
half the CUs.  Each case checks the schedule named, then runs AUTO -- which from
33 rows takes another tile of its own on most of them (hipgemm_auto_tile) --
and the named schedule itself, through the plain entry point (a workspace
allocated for the call where one is needed) and through the workspace entry
point, on ternary inputs (every sum exact): all must equal the oracle bit for
bit.  AUTO comes back to the split-K schedule where its tiles are not built: an
extended epilogue without aligned stores.
"""
import numpy as np
import pytest

import hipgemm_amd as hg
from util import from_dev_bf16, say, scale_tensor, to_dev

pytestmark = pytest.mark.gpu

V = hg.VARIANTS
TERNARY = np.array([0xB8, 0x00, 0x38], np.uint8)  # -1, 0, +1


CASES = [
    (64, 4096, 4096, "strip"),      # 32-column strips, 2 K-slices
    (40, 2048, 8192, "strip"),      # 4 K-slices
    (33, 6144, 2048, "strip"),      # 192 strips, one K-slice
    (48, 3072, 8192, "strip"),      # 64-column strips fill the CUs better
    (40, 14336, 8192, "strip"),     # 64-column strips: 448 of 32 > CUs
    (64, 8192, 8192, "strip"),
    (16, 28672, 8192, "strip"),     # up to 16 rows: strips throughout
    (32, 28672, 8192, "tile128"),   # N > 64 x CUs from 17 rows
    (28, 20480, 1536, "tile128"),
    (40, 24576, 8192, "tile128"),
    (56, 8192, 14336, "tile128"),   # above 48 rows, K > 8192
    (48, 8192, 14336, "strip"),     # three 16-row blocks
    (40, 3072, 1024, "strip"),      # K <= 1024, 96 strips
    (40, 2048, 1024, "tile128"),    # ... 64 strips
    (96, 2048, 4096, "strip"),      # 65-128 rows, B_T of at most 8 MiB
    (128, 6144, 2048, "tile128"),   # half-filled, but 2 slices
    (120, 2560, 4096, "skinny"),    # half-filled, 4 slices
    (100, 4096, 4096, "skinny"),
    (1536, 4096, 4096, "tile128"),  # 96 tiles of 256, 384 of 128
    (1152, 4096, 4096, "tile128"),
    (640, 8192, 4096, "4wave_mfma16"),   # the same region, a side of 8192
    (2048, 4096, 4096, "4wave_mfma16"),  # 512 tiles of 128: two full rounds
]


@pytest.mark.parametrize("M,N,K,pick", CASES)
def test_auto_pick_bit_exact(gpu, oracle, M, N, K, pick):
    torch = gpu
    say(f"case auto-pick M={M} N={N} K={K} want={pick} seed=17")
    assert hg.select_variant(M, N, K) == V[pick]
    check(torch, oracle, M, N, K, 0)


@pytest.mark.parametrize("M,N,K,pick", CASES)
def test_named_schedule_bit_exact(gpu, oracle, M, N, K, pick):
    say(f"case auto-named M={M} N={N} K={K} variant={pick} seed=17")
    check(gpu, oracle, M, N, K, V[pick])


# The tile that AUTO runs in place of the schedule it names, on 256 CUs.
OWN = {(64, 4096, 4096): (64, 64), (48, 3072, 8192): (64, 64),
       (64, 8192, 8192): (64, 64), (56, 8192, 14336): (128, 64),
       (40, 3072, 1024): (64, 64), (40, 2048, 1024): (64, 64),
       (96, 2048, 4096): (64, 64), (128, 6144, 2048): (64, 64),
       (120, 2560, 4096): (64, 64), (100, 4096, 4096): (64, 64),
       (1536, 4096, 4096): (192, 128), (1152, 4096, 4096): (192, 128),
       (640, 8192, 4096): (192, 128), (2048, 4096, 4096): (128, 256)}


@pytest.mark.parametrize("M,N,K,pick", CASES)
def test_auto_own_tile(M, N, K, pick):
    assert hg.auto_tile(M, N, K) == OWN.get((M, N, K))


@pytest.mark.parametrize("ws", [False, True], ids=["allocated", "workspace"])
def test_auto_split_k_where_its_tiles_are_not_built(gpu, oracle, ws):
    """bf16 with a bias and an odd ldc: 2-byte stores, which 64-column tiles have
    for the plain epilogue only, so that AUTO runs the schedule it names."""
    torch = gpu
    M, N, K = 100, 4095, 4096
    say(f"case auto split-K fallback M={M} N={N} K={K} workspace={ws}")
    assert hg.select_variant(M, N, K) == V["skinny"] and hg.auto_tile(M, N, K)
    rng = np.random.default_rng(18)
    A = TERNARY[rng.integers(0, 3, (M, K))]
    B = TERNARY[rng.integers(0, 3, (N, K))]
    bias = rng.uniform(-4, 4, N).astype(np.float32)
    a, b, v = to_dev(torch, A), to_dev(torch, B), torch.from_numpy(bias).cuda()
    c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    d = hg.GemmDesc(A=a.data_ptr(), B_T=b.data_ptr(), C=c.data_ptr(), M=M, N=N, K=K,
                    lda=K, ldb=K, ldc=N, bias=v.data_ptr())
    if ws:
        w = torch.zeros(hg.workspace_size(M, N, K, 0), dtype=torch.uint8, device="cuda")
        d.workspace, d.workspace_bytes = w.data_ptr(), w.numel()
    assert hg.gemm_desc_raw(d, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert np.array_equal(from_dev_bf16(c), oracle.gemm_ex(A, B, bias=bias))


def check(torch, oracle, M, N, K, variant):
    rng = np.random.default_rng(17)
    A = TERNARY[rng.integers(0, 3, (M, K))]
    B = TERNARY[rng.integers(0, 3, (N, K))]
    want = oracle.gemm(A, B, 0.5, 2.0)
    a, b = to_dev(torch, A), to_dev(torch, B)
    sa, sb = scale_tensor(torch, 0.5), scale_tensor(torch, 2.0)
    stream = torch.cuda.current_stream().cuda_stream
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert hg.gemm_raw(a.data_ptr(), b.data_ptr(), out.data_ptr(), M, N, K, K,
                       K, N, sa.data_ptr(), sb.data_ptr(), variant, stream) == 0
    torch.cuda.synchronize()
    got = from_dev_bf16(out)
    assert np.array_equal(got, want), (
        f"plain entry: {int((got != want).sum())} of {M * N} outputs differ")
    need = hg.workspace_size(M, N, K, variant)
    ws = torch.zeros(max(need, 256), dtype=torch.uint8, device="cuda")
    out.fill_(float("nan"))
    assert hg.gemm_raw_ws(a.data_ptr(), b.data_ptr(), out.data_ptr(), M, N, K,
                          K, K, N, sa.data_ptr(), sb.data_ptr(), variant,
                          ws.data_ptr(), need, stream) == 0
    torch.cuda.synchronize()
    got = from_dev_bf16(out)
    assert np.array_equal(got, want), (
        f"workspace entry: {int((got != want).sum())} of {M * N} outputs differ")
    if need:
        assert not ws[:16384].cpu().numpy().any(), "counters not left zero"


def test_sweep_module_reports_auto(gpu):
    """hipgemm_amd.sweep times the schedules that take a shape and reports
    AUTO's pick against the fastest (measurement only)."""
    import io

    from hipgemm_amd import sweep

    say("case sweep 64x1024x1024 strip/tile128, 128x256x256 all")
    buf = io.StringIO()
    r = sweep.sweep([(64, 1024, 1024), (128, 256, 256)], [V["strip"], V["tile128"], V["skinny"]],
                    rounds=2, launches=10, out=buf)
    text = buf.getvalue()
    assert len(r) == 2 and all(x >= 1.0 for x in r), text
    assert "64x1024x1024:" in text and "summary: 2 shapes" in text
