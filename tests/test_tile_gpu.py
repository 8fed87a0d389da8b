"""AUTO's tiles other than its schedules' own (hipgemm_auto_tile): where AUTO
takes them, and their results against the oracle, bit for bit on ternary
operands (every partial sum exact, in any order).

Shapes end inside a tile in both directions, inside a K-step, or exactly on
them, run one and several tiles per workgroup, and take 16-byte stores of C or
not; every output type and epilogue option of the general entry point runs on
every tile, with canaries around C.  64-column tiles split K where the call
brings a workspace: every call runs without one, and twice with one, whose
counters have to end at zero.
"""
import numpy as np
import pytest

import hipgemm_amd as hg
from oracle import pyoracle as po
from util import say, to_dev

TERN = {0: np.array([0xB8, 0x00, 0x38], np.uint8),
        1: np.array([0xBC, 0x00, 0x3C], np.uint8)}
ES = {po.OUT_BF16: 2, po.OUT_F16: 2, po.OUT_F32: 4, po.OUT_FP8: 1}
NP = {4: np.uint32, 2: np.uint16, 1: np.uint8}

# shape -> AUTO's tile on 256 CUs
SHAPES = {
    (64, 8192, 8192): (64, 64),      # 2 K-slices
    (33, 200, 4096): (64, 64),       # 8 K-slices
    (127, 1001, 4112): (64, 64),     # odd N; K ends inside a step
    (128, 8192, 8192): (128, 64),    # 2 K-slices
    (65, 9000, 1040): (128, 64),
    (144, 256, 2272): (64, 64),      # ragged rows of tiles, K-slices
    (300, 1000, 4112): (64, 64),
    (200, 6144, 640): (128, 64),
    (700, 1501, 528): (128, 64),     # odd N: 2-byte stores
    (1163, 206, 2112): (128, 128),   # K-split plan, run unsplit
    (4221, 1832, 16): (128, 128),    # two rounds, one K-step
    (2055, 3640, 336): (128, 256),
    (1201, 5891, 240): (128, 256),   # odd N
    (4367, 4672, 144): (128, 256),   # several tiles per workgroup
    (2304, 3840, 512): (192, 192),   # whole tiles and steps
    (1865, 4391, 144): (192, 192),   # odd N
    (4051, 4416, 432): (192, 192),   # several tiles per workgroup
    (1237, 3280, 592): (192, 128),
    (1537, 5392, 1040): (192, 128),  # several tiles per workgroup
    (2119, 4149, 16): (192, 128),    # odd N, two rounds, one K-step
    (2304, 2304, 1024): (192, 128),  # whole tiles and steps
    (107, 17832, 32): (128, 64),     # one row of more tiles than workgroups:
    (72, 20648, 128): (128, 64),     # on whole lines of B_T, each read once
    (77, 17849, 16): (128, 64),      # odd N
}


def tiles_of(shape):
    (M, N, _), (bm, bn) = shape, SHAPES[shape]
    return -(-M // bm) * -(-N // bn)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_auto_tile(shape):
    M, N, K = shape
    assert hg.auto_tile(M, N, K) == SHAPES[shape]
    assert hg.split_columns(M, N, K) == 0


def test_shapes_cover_one_and_several_tiles_per_workgroup():
    """(AUTO runs 64 x 64 tiles in one round only.)"""
    for tile in set(SHAPES.values()):
        n = [tiles_of(s) for s in SHAPES if SHAPES[s] == tile]
        assert min(n) <= 256 and (max(n) > 256) == (tile != (64, 64)), tile


def test_one_row_of_64_column_tiles_in_one_round():
    """Where 128 x 128 tiles are named, more 64-column tiles than CUs in one row
    are not taken; where strips are, they may be."""
    for M in (33, 48, 64):
        for N in (16448, 17408, 24576, 32768):
            for K in (1024, 4096, 8208, 11008):
                assert hg.select_variant(M, N, K) == hg.VARIANTS["tile128"]
                assert hg.auto_tile(M, N, K) is None, (M, N, K)
    assert hg.select_variant(107, 17832, 32) == hg.VARIANTS["strip"]


def test_auto_tile_keeps_other_choices():
    """None up to 32 rows, where 256 x 256 tiles fill whole rounds, for the
    documented column split, or without work."""
    for M, N, K in [(32, 8192, 8192), (16, 4096, 4096), (8192, 8192, 8192),
                    (4096, 4096, 4096), (8192, 28672, 8192), (4000, 5000, 3584),
                    (300, 300, 0), (0, 64, 64)]:
        assert hg.auto_tile(M, N, K) is None, (M, N, K)


def test_short_workspace_is_refused():
    """Whichever tile runs, AUTO refuses a workspace too small for the schedule
    that hipgemm_select_variant names (before any launch); in these shapes that
    schedule needs all of hipgemm_workspace_size."""
    fake = 1 << 20
    for M, N, K in SHAPES:
        need = hg.workspace_size(M, N, K, 0)
        if need:
            assert hg.gemm_raw_ws(fake, fake, fake, M, N, K, K, K, N, 0, 0, 0, fake,
                                  need - 256) == hg.hipErrorInvalidValue


def run(torch, A, B, out, ldc, *, fb=0, act=0, sa=None, sr=None, sc=None, bias=None,
        so=None, ws=None):
    M, K = A.shape
    N = B.shape[0]
    es = ES[out]
    dev = {k: None if v is None else torch.from_numpy(
        np.ascontiguousarray(v, np.float32).reshape(-1)).to("cuda")
        for k, v in dict(sa=sa, sr=sr, sc=sc, bias=bias, so=so).items()}
    ptr = {k: v.data_ptr() if v is not None else 0 for k, v in dev.items()}
    a, b = to_dev(torch, A), to_dev(torch, B)
    buf = torch.full(((M + 4) * ldc * es,), 0xA5, dtype=torch.uint8, device="cuda")
    d = hg.GemmDesc(A=a.data_ptr(), B_T=b.data_ptr(), C=buf.data_ptr() + 2 * ldc * es,
                    M=M, N=N, K=K, lda=K, ldb=K, ldc=ldc, b_format=fb,
                    out_dtype=out, activation=act, scale_a=ptr["sa"],
                    scale_rows=ptr["sr"], scale_cols=ptr["sc"], bias=ptr["bias"],
                    scale_out=ptr["so"],
                    workspace=0 if ws is None else ws.data_ptr(),
                    workspace_bytes=0 if ws is None else ws.numel())
    assert hg.gemm_desc_raw(d, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    got = buf.cpu().numpy().reshape(M + 4, ldc * es)
    guard = (np.all(got[:2] == 0xA5) and np.all(got[M + 2:] == 0xA5) and
             np.all(got[2:M + 2, N * es:] == 0xA5))
    C = np.ascontiguousarray(got[2:M + 2, :N * es]).view(NP[es])
    return C, guard


def runs(torch, A, B, out, ldc, want, **kw):
    """Without a workspace, then twice with one."""
    M, K = A.shape
    need = hg.workspace_size(M, B.shape[0], K, 0)
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda") if need else None
    for w in (None, ws, ws) if need else (None,):
        C, guard = run(torch, A, B, out, ldc, ws=w, **kw)
        assert guard, "write outside M x N"
        assert np.array_equal(C, want), f"{int((C != want).sum())} of {C.size} differ"
        assert w is None or not w[:16384].cpu().numpy().any(), "counters not left zero"


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_tile_bit_exact(gpu, oracle, shape):
    M, N, K = shape
    rng = np.random.default_rng(5)
    for fb, pad in ((0, 0), (1, 8), (0, 3)):  # ldc = N + 3: 2-byte stores
        say(f"case tile {SHAPES[shape]} M={M} N={N} K={K} fb={fb} ldc=N+{pad}")
        A = TERN[0][rng.integers(0, 3, (M, K))]
        B = TERN[fb][rng.integers(0, 3, (N, K))]
        want = oracle.gemm_ex(A, B, b_fmt=fb, scale_a=0.5)
        runs(gpu, A, B, po.OUT_BF16, N + pad, want, fb=fb, sa=[0.5])


@pytest.mark.gpu
@pytest.mark.parametrize("out", [po.OUT_BF16, po.OUT_F16, po.OUT_F32, po.OUT_FP8],
                         ids=["bf16", "f16", "f32", "e4m3"])
@pytest.mark.parametrize("shape", [s for s in SHAPES if s[1] % 8 == 0],
                         ids=lambda s: "x".join(map(str, s)))
def test_tile_epilogue(gpu, oracle, shape, out):
    M, N, K = shape
    rng = np.random.default_rng(6)
    A, B = TERN[0][rng.integers(0, 3, (M, K))], TERN[1][rng.integers(0, 3, (N, K))]
    sr = np.exp2(rng.integers(-3, 4, M)).astype(np.float32)
    sc = np.exp2(rng.integers(-3, 4, N)).astype(np.float32)
    bias = rng.uniform(-4, 4, N).astype(np.float32)
    so = 0.25 if out == po.OUT_FP8 else None
    for act in (po.ACT_NONE, po.ACT_RELU):
        say(f"case tile {SHAPES[shape]} M={M} N={N} K={K} out={out} act={act}")
        want = oracle.gemm_ex(A, B, b_fmt=1, out=out, act=act, scale_a=0.5,
                              scale_rows=sr, scale_cols=sc, bias=bias,
                              scale_out=so or 1.0)
        runs(gpu, A, B, out, N + 8, want, fb=1, act=act, sa=[0.5], sr=sr, sc=sc,
             bias=bias, so=None if so is None else [so])


# Largest step between neighbouring values, relative, and the smallest value that
# it holds down to.
STEP = {po.OUT_BF16: (2.0 ** -7, 2.0 ** -126), po.OUT_F16: (2.0 ** -10, 2.0 ** -14),
        po.OUT_F32: (1e-5, 0.0), po.OUT_FP8: (2.0 ** -3, 2.0 ** -6)}


def values(torch, bits, out):
    dt = {po.OUT_BF16: torch.bfloat16, po.OUT_F16: torch.float16,
          po.OUT_F32: torch.float32, po.OUT_FP8: torch.float8_e4m3fn}[out]
    return torch.from_numpy(bits.view({4: np.int32, 2: np.int16, 1: np.uint8}[ES[out]])
                            ).view(dt).double().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("act", [po.ACT_SILU, po.ACT_GELU_TANH], ids=["silu", "gelu"])
@pytest.mark.parametrize("shape", [
    (33, 200, 4096), (200, 6144, 640), (72, 20648, 128), (4221, 1832, 16),
    (2055, 3640, 336), (2304, 3840, 512), (1237, 3280, 592)],
    ids=lambda s: "x".join(map(str, s)))
def test_tile_transcendental(gpu, oracle, shape, act):
    """silu and gelu on every tile and output type.  The values before the
    activation are exact; it is evaluated with an exponential of relative error
    2^-24 |log2| (|log2| < 100 here) and a reciprocal: fp32 within 1e-5, the other
    types at most one step apart, and equal but for values that close to a
    midpoint (1e-5 of 2^-8 at the most: under 1 %).  2^-46 for the oracle's 1 +
    tanh, which cancels in double precision (|v| 2^-52, |v| < 2^6)."""
    M, N, K = shape
    rng = np.random.default_rng(9)
    A, B = TERN[0][rng.integers(0, 3, (M, K))], TERN[0][rng.integers(0, 3, (N, K))]
    sa = 2.0 ** -round(np.log2(K ** 0.5 * 0.5))  # standard deviation about 1.3
    bias = rng.integers(-8, 9, N).astype(np.float32) / 8
    need = hg.workspace_size(M, N, K, 0)
    for out in ES:
        say(f"case tile {SHAPES[shape]} M={M} N={N} K={K} out={out} act={act}")
        so = 4.0 if out == po.OUT_FP8 else None
        want = oracle.gemm_ex(A, B, out=out, act=act, scale_a=sa, bias=bias,
                              scale_out=so or 1.0)
        r = values(gpu, want, out)
        for ws in (0, need) if need else (0,):
            w = gpu.zeros(ws, dtype=gpu.uint8, device="cuda") if ws else None
            C, guard = run(gpu, A, B, out, N + 8, act=act, sa=[sa], bias=bias,
                           so=None if so is None else [so], ws=w)
            assert guard, "write outside M x N"
            step, least = STEP[out]
            c = values(gpu, C, out)
            assert np.all(np.abs(c - r) <= step * np.maximum(np.abs(r), least) + 2.0 ** -46)
            assert out == po.OUT_F32 or np.mean(C == want) > 0.99


@pytest.mark.gpu
@pytest.mark.parametrize("tail", [0, 16, 112])
def test_each_xcd_starts_at_its_own_step(gpu, tail):
    """Workgroups on different XCDs walk K from different steps, also where K
    ends inside a step.  Step 0 adds 2^23 and every other one 0.5, which is
    lost on top of that, so the fp32 sum grows with the steps that came before
    step 0; every tile (one per workgroup) has the same operands."""
    torch = gpu
    M, N, K = 128, 128 * 32, 8 * 128 + tail
    say(f"case start steps tile128 M={M} N={N} K={K}")
    A, B = np.full((M, K), 0x38, np.uint8), np.zeros((N, K), np.uint8)
    A[:, :128] = B[:, :128] = 0x78  # 256 * 256 * 128 = 2^23
    B[:, 128::128] = 0x30           # 1 * 0.5
    a, b = to_dev(torch, A), to_dev(torch, B)
    c = hg.gemm(a, b, out_dtype=torch.float32, variant=hg.VARIANTS["tile128"])
    tiles = c.cpu().numpy().reshape(M, 32, 128)
    sums = tiles[0, :, 0]
    assert np.all(tiles == sums[None, :, None])
    assert np.all((sums >= 2.0 ** 23) & (sums <= 2.0 ** 23 + 4)), sums
    assert len(set(sums)) > 1, sums


@pytest.mark.gpu
@pytest.mark.parametrize("shape,split", [((128, 2048, 8192), True),
                                         ((79, 2560, 4096), False)])
def test_split_k_where_outputs_take_no_slices(gpu, shape, split):
    """AUTO names the split-K schedule at both shapes.  bf16 outputs run K-slices
    of 64-column tiles; fp32 outputs, which have none, run the schedule itself
    or whole K, whichever is faster.  The fp32 sums tell which ran (their results are
    checked where sums are exact)."""
    torch = gpu
    M, N, K = shape
    say(f"case split-K or whole K M={M} N={N} K={K} fp32 output")
    skinny = hg.VARIANTS["skinny"]
    assert hg.select_variant(M, N, K) == skinny and hg.auto_tile(M, N, K)[1] == 64
    rng = np.random.default_rng(8)  # every finite e4m3 value: inexact sums
    a, b = (to_dev(torch, rng.integers(0, 127, s, np.uint8) |
                   rng.integers(0, 2, s, np.uint8) << 7) for s in ((M, K), (N, K)))
    f32 = torch.float32
    auto = hg.gemm(a, b, out_dtype=f32)
    named = hg.gemm(a, b, out_dtype=f32, variant=skinny)
    assert torch.equal(auto, named) == split
