"""Which products a step of few rows takes, seen on the CPU, before anything is launched: in attention through a latent the first product that the layer
asks for stands for the route."""
import types

import pytest
import torch

from inferflux_amd.kernels import ops
from inferflux_amd.parts.latent_attention import LatentAttention
from inferflux_amd.parts.plan import PartSpec

BF16 = torch.bfloat16


class Asked(Exception):
    pass


def tiled(rows):
    """A weight with a copy, of which only its existence is looked at here."""
    return ops.LinearWeight(rows, torch.empty(0, dtype=rows.dtype), None, ops.choose_tile_rows(rows.shape[0]))


def route(monkeypatch, hidden, rows, q_rank, gate, requests):
    """("joined" | "normed" | "apart", whether partial sums are taken) of a step of ``rows`` plain rows of ``requests`` requests."""
    a = LatentAttention("a", hidden, 8, 64, 32, 64, q_rank, 96, 0.1, 1e-5, PartSpec("none"), output_gate=gate)
    zeros = lambda *shape: torch.zeros(shape, dtype=BF16)
    a.load({n: zeros(*s.shape) for n, s in a.param_specs().items()})
    a.w_down, a.w_uq = tiled(a.w_down.rows), tiled(a.w_uq.rows)
    if q_rank:
        a.few_scale = torch.ones(a.w_down.shape[0], dtype=BF16)
    elif not gate:
        a.w_few = tiled(torch.cat([a.w_uq.rows, a.w_down.rows]))
    a.position = types.SimpleNamespace(kernel_args=lambda ctx: (None, 0, None, None))

    def linear(x, weight, out_dtype=None, keep_slices=False):
        raise Asked("joined" if weight is a.w_few else "apart", keep_slices and ops.ring_takes_few(x, weight, True) == 2)

    def normed(*args):
        raise Asked("normed", False)
    monkeypatch.setattr(ops, "linear", linear)
    monkeypatch.setattr(ops, "linear_normed", normed)
    cache = types.SimpleNamespace(group=0, k=zeros(1, 1, 16, 128))
    ctx = types.SimpleNamespace(timer=None, write_slots=lambda group: None, n_tokens=rows, n_requests=requests)
    with pytest.raises(Asked) as asked:
        a.forward(zeros(rows, hidden), ctx, types.SimpleNamespace(cache=cache, writes_cache=True))
    return asked.value.args


@pytest.mark.parametrize("rows", [1, 8, 9, 12, 16])
@pytest.mark.parametrize("q_rank,gate", [(768, False), (768, True), (None, False)])
@pytest.mark.parametrize("hidden", [2048, 4088, 4096, 5120])
def test_down_products_whose_sums_stayed_in_float_still_do(monkeypatch, hidden, q_rank, gate, rows):
    """9 to 16 plain rows times a deep down projection go to the ring in slices of K, whose float sums the latent's norm, the rotation and the
    output gate's sigmoid read: neither of the joined products, which write bfloat16, may take them away."""
    deep = rows >= 9 and hidden >= 4096
    assert route(monkeypatch, hidden, rows, q_rank, gate, rows) == ("apart" if deep else "normed" if q_rank else "joined", deep)
    if rows > 1:         # a prompt
        assert route(monkeypatch, hidden, rows, q_rank, gate, 1) == ("apart" if deep or q_rank else "joined", deep)


@pytest.mark.parametrize("N,K", [(8, 4096), (2048, 4096), (2048, 4088), (2048, 4104), (2052, 4096), (896, 4864), (8, 1 << 20), (16, (1 << 20) - 8), (64, 4100)])
def test_what_is_not_added_into_the_stream_leaves_its_sums_in_float(N, K):
    """``adds_into_stream`` gives a product to the norm only where ``linear`` then leaves partial sums: a rounded one would lose what the stream's
    epilogue keeps."""
    weight, norm = tiled(torch.empty((N, K), dtype=BF16)), torch.empty(N, dtype=BF16)
    for rows in (8, 9, 16):
        x = torch.empty((rows, K), dtype=BF16)
        into, sums = ops.adds_into_stream(rows, weight, norm), ops.ring_takes_few(x, weight, True) == 2
        assert into or sums or K % 8, (rows, N, K)
        assert into == (not sums or N > 2048) or K % 8, (rows, N, K)
    assert ops.adds_into_stream(16, ops.LinearWeight(weight.rows), norm) == (K % 8 == 0)
