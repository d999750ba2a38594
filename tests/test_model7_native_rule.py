"""Which calls the native stack takes, by sizes alone: the rule looks at shapes and places, so expanded tensors of one value do."""
import pytest
import torch


def case(B, T, C, d=32, L=1):
    from jaxrwkv_amd import blocks7
    one = torch.zeros(1, dtype=torch.bfloat16)
    shapes = {"r_k": (L, C // 64, 64), "ffn_key": (L, 4 * C, C), "ffn_value": (L, C, 4 * C)}
    shapes.update({n: (L, C, C) for n in ("receptance", "key", "value", "output")})
    for f in "wavg":
        shapes.update({f + "1": (L, C, d), f + "2": (L, d, C)})
    params = [one.expand(shapes.get(n, (L, C))) for n in blocks7.NAMES]
    state = torch.zeros((B, L, 66, C), dtype=torch.bfloat16)
    return blocks7._native(params, one.expand(B, T, C), state, False)


@pytest.mark.parametrize("B,T,C,native", [
    (4, 512, 768, True), (4, 2048, 768, True), (8, 1000, 1024, True), (4, 600, 1536, True), (4, 250, 2048, True), (1, 250, 4096, True),
    (1, 1400, 2048, False), (4, 550, 2048, False), (4, 625, 2048, False), (4, 675, 2048, False), (4, 1021, 2048, False), (1, 600, 4096, False),
    (4, 1200, 1536, False), (9, 1000, 768, False)])
def test_sizes(B, T, C, native):
    """Where the separate steps' library products were measured faster (2048 channels: 2200 rows forward 11.6 ms against 12.9), or the
    workspace would be large, the call takes them."""
    assert case(B, T, C) == native


@pytest.mark.parametrize("B,T,C,d,native", [(1, 9, 128, 2 ** 20, True), (1, 9, 128, 2 ** 22, False), (4, 512, 768, 2 ** 19, False), (1, 9, 128, 12, False)])
def test_inner_sizes(B, T, C, d, native):
    """What the native code refuses (operands of 2 GiB, sizes that are no multiple of 8) takes the separate steps."""
    assert case(B, T, C, d) == native
