"""The K mean of a re-quantised chunk where its route changes: chunks of at most 32 blocks form it inside the quantiser,
longer ones in the finaliser, with 16 or 32 channels a workgroup. Every ring field bit for bit against the oracle, in
both input formats, also through the prologue (which quantises V in the last pass)."""
import pytest
import torch

from oracle import emu
from oracle import prologue as pro

pytestmark = pytest.mark.gpu

DEV = "cuda"
# 29 .. 32 blocks fill the last super-block of the in-quantiser form; 2049 tokens are 33 blocks, the finaliser's first
EDGES = [1793, 1984, 1985, 2048, 2049, 2112]


def _k():
    from lingbot_world_v2_realtime_amd import kernels
    return kernels


def _check(ring, layer, ref, n):
    nb = (n + 63) // 64
    for name in ("km", "k_scale", "k8", "v8", "v8lo", "v_scale"):
        got = getattr(ring, name)[layer, 0].cpu()
        got = got if name == "km" else got[:, :nb * 64] if name == "k8" else got[:, :nb]
        assert torch.equal(got, ref[name]), name


def _kv(shape, h, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    k = torch.randn(*shape, h, 128, generator=g) + 3 * torch.randn(*shape[:-1], 1, h, 128, generator=g)
    return k.to(dtype), (torch.randn(*shape, h, 128, generator=g) * 1.7).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", EDGES)
def test_requant_mean_edges(n, dtype):
    k, v = _kv((1, n), 2, dtype, n)
    ring = _k().RingCache(1, 1, 2, _k().pad_to(n, 64), 1, DEV)
    _k().kv_requant(k.to(DEV), v.to(DEV), ring, 0)
    torch.cuda.synchronize()
    _check(ring, 0, emu.requant(k, v), n)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layers", [31, 32])
def test_requant_finaliser_widths(layers, dtype):
    """4 heads: 31 layers are 124 (head, layer) pairs, below the 128 from which the finaliser is 32 channels wide."""
    n = 2049
    k, v = _kv((layers, 1, n), 4, dtype, layers)
    ring = _k().RingCache(layers, 1, 4, _k().pad_to(n, 64), 1, DEV)
    _k().kv_requant(k.to(DEV), v.to(DEV), ring, 0)
    torch.cuda.synchronize()
    for layer in (0, 17, layers - 1):
        _check(ring, layer, emu.requant(k[layer], v[layer]), n)


@pytest.mark.parametrize("n", [1985, 2048, 2049])
def test_prologue_mean_edges(n):
    from lingbot_world_v2_realtime_amd.layers.prologue import ChunkRope, rope_freqs
    h, g = 2, torch.Generator().manual_seed(n)
    x = (torch.randn(1, n, h * 128, generator=g) + 3 * torch.randn(1, 1, h * 128, generator=g)).bfloat16()
    v = (torch.randn(1, n, h, 128, generator=g) * 1.7).bfloat16()
    w = (1 + 0.3 * torch.randn(h * 128, generator=g)).bfloat16()
    ring = _k().RingCache(1, 1, h, _k().pad_to(n, 64), 1, DEV)
    k_out = _k().norm_rope_kv_requant(x.to(DEV), v.to(DEV), h, w.to(DEV), 1e-6, ChunkRope(rope_freqs(DEV), 20, 26, 3),
                                      ring, 0)
    torch.cuda.synchronize()
    roped = pro.norm_rope(x[0], w, 1e-6, h, pro.rope_table(), (20, 26), 3)
    assert torch.equal(k_out[0].cpu(), roped)
    _check(ring, 0, emu.requant(roped, v[0]), n)
