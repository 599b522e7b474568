"""A step's largest probability, where it is the largest so far, is exactly 1: probabilities that are rounded to 16 bits as they
are (16-bit pages, FP8 pages of one multiplier a head) lose nothing there. Two keys that outweigh all others, the larger
in a later step of the same wavefront, weigh as float64 has it to FP32's precision."""
import pytest
import torch

from tests.support import Cache

pytestmark = pytest.mark.gpu
dev = "cuda"

# Scores below 10 in log2 units, rounded at 2^-21; the exponential, the factor and three sums at 2^-24 each: 2e-6 of values
# up to 5. A rounded weight between 1/2 and 1 is off by up to 2^-9 of it: 1e-3 and more over these heads.
ATOL = 2e-5


@pytest.mark.parametrize("kind,hkv,g,d", [("bf16", 2, 4, 128), ("bf16", 3, 4, 128), ("fp16", 2, 4, 128), ("bf16", 2, 4, 256), ("bf16", 4, 4, 64),
                                          ("fp8", 2, 4, 128), ("fp8", 3, 4, 128), ("fp8", 2, 4, 256), ("fp8", 4, 4, 64)])
@pytest.mark.parametrize("columns", [1, 4, 5, 8])      # one query tile to four
@pytest.mark.parametrize("gap", [32, 64])              # the next step of the same wavefront: of two heads' tiles, of one's
@pytest.mark.parametrize("fused", [False, True])
def test_two_steps_largest_probabilities_are_exact(kind, hkv, g, d, columns, gap, fused):
    n = 200
    cache = Cache(kind, hkv, d, d, 16, [n], multipliers=(1.0, 1.0))
    keys = torch.zeros(n, hkv, d, device=dev)
    keys[:, :, 0] = -64.0
    keys[3, :, 0], keys[3 + gap, :, 0] = 4.0, 4.5
    cache.write(0, 0, keys, torch.randn(n, hkv, d, generator=torch.Generator().manual_seed(d)).to(dev))
    q = torch.zeros(columns, hkv * g, d, device=dev)
    q[:, :, 0] = 0.25 + torch.arange(columns * hkv * g, device=dev).view(columns, -1) % 21 / 16
    out = torch.empty(columns, hkv * g, d, device=dev)
    cache.attend(q, [0], [0], [n - columns], columns, scale=1.0, out=out, fused=fused)
    want, _ = cache.want(q, 0, n - columns, columns, scale=1.0)
    assert float((out.double().cpu() - want).abs().max()) < ATOL
