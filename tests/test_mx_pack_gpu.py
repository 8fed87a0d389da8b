"""hipgemm_mx_pack_scales on sources and packed buffers of every alignment, with
canaries around the packed buffer: equal to the packing of a contiguous copy
(whose layout test_mx_gpu.py checks)."""
import pytest

import hipgemm_amd as hg
from util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,K", [(1, 32), (130, 256), (128, 288), (300, 2048),
                                    (257, 8192 + 32)])
@pytest.mark.parametrize("pad,off,doff", [(0, 0, 0), (8, 8, 0), (3, 0, 0), (0, 1, 0),
                                          (8, 0, 1), (5, 3, 7), (3, 4, 0), (7, 4, 16)])
def test_pack_alignments(gpu, rows, K, pad, off, doff):
    torch = gpu
    say(f"case mx-pack rows={rows} K={K} ld=K/32+{pad} src+{off} dst+{doff}")
    kb, ld = K // 32, K // 32 + pad
    src = torch.randint(0, 256, (rows * ld + off,), dtype=torch.uint8, device="cuda")
    view = src[off:].view(rows, ld)[:, :kb]
    n = hg.mx_scales_bytes(rows, K)
    buf = torch.full((n + 64 + doff,), 0xA5, dtype=torch.uint8, device="cuda")
    assert hg.lib().hipgemm_mx_pack_scales(
        view.data_ptr(), rows, K, ld, buf.data_ptr() + 32 + doff,
        torch.cuda.current_stream().cuda_stream or None) == 0
    want = hg.mx_pack_scales(view.contiguous(), K)
    torch.cuda.synchronize()
    assert torch.equal(buf[32 + doff:32 + doff + n], want[:n])
    assert bool((buf[:32 + doff] == 0xA5).all()) and bool((buf[32 + doff + n:] == 0xA5).all())
