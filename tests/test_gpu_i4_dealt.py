"""The int8 kernel of short launches with one scale per row, whose waves share out the groups of a stage: rows and channels that end
inside a tile, K from the shortest ring on and with a last stage that repeats one, two or three groups, both ring depths and
all three tiles, several weight matrices, a residual -- against the 64 x 64 tiles of four waves, which the parity tests pin to the oracle."""
import numpy as np
import pytest

from flh_amd import synthetic as syn

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("k", [512, 640, 768, 896, 1408, 2688])
@pytest.mark.parametrize("m,ns", [(1, (12416,)), (16, (12544, 72)), (17, (8,)), (17, (136, 40)), (32, (1000, 24)), (33, (264,)), (63, (8200,)),
                                  (64, (4096, 1024, 1024)), (65, (4104,)), (130, (4096,)), (300, (136,)), (1280, (72,)), (64, (14336,)),
                                  (97, (8200, 24))])
def test_against_the_square_tiles(gemm_tuning, m, ns, k):
    """(The last two: more than 768 blocks of 32 x 32, which take the tile of 64 tokens.)"""
    against_the_square_tiles(gemm_tuning, m, ns, k)


@pytest.mark.parametrize("m,ns,k", [(64, (8192,), 8320), (33, (8160, 8), 8448), (100, (4064,), 8576)])
def test_long_rows(gemm_tuning, m, ns, k):
    """K beyond 8192 with 257 .. 512 blocks of 32 x 32 and at most 256 of 64 x 32: the tile of 64 tokens again."""
    columns = -(-sum(ns) // 32)
    assert 256 < -(-m // 32) * columns <= 512 and -(-m // 64) * columns <= 256
    against_the_square_tiles(gemm_tuning, m, ns, k)


def against_the_square_tiles(gemm_tuning, m, ns, k):
    from flh_amd import _ops as ops
    rng = np.random.default_rng(m + k)
    a, sa = dev(rng.integers(0, 256, size=(m, k // 2), dtype=np.uint8)), dev(syn.weight_scales(m, 1, m))
    ws = [dev(rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)) for n in ns]
    sw = [dev(syn.weight_scales(n, 1, n)) for n in ns]
    res = dev(rng.standard_normal((m, ns[0])).astype(np.float16))

    def run():
        return [*ops.gemm_i4_dequant_multi(a, ws, sa, sw, k), ops.gemm_i4_dequant_add(a, ws[0], sa, sw[0], res, k)]
    got = run()
    gemm_tuning(64, 1)
    for i, (x, y) in enumerate(zip(got, run())):
        assert torch.equal(x, y), i


@pytest.mark.parametrize("m", [5, 40, 100])
def test_odd_channels_and_largest_sums(m):
    """All codes -8: every product is 64, the sum 64 K; channels that are no multiple of four."""
    from flh_amd import _ops as ops
    n, k = 4099, 1024
    a, w = torch.full((m, k // 2), 0x88, dtype=torch.uint8, device="cuda"), torch.full((n, k // 2), 0x88, dtype=torch.uint8, device="cuda")
    sa, sw = torch.full((m, 1), 2.0 ** -4, device="cuda").half(), torch.full((n, 1), 2.0 ** -6, device="cuda").half()
    assert torch.equal(ops.gemm_i4_dequant(a, w, sa, sw, k), torch.full((m, n), 64.0 * k / 1024, device="cuda").half())
