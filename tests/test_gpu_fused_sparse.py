"""Layers with tensors of k < 1024 through the fused launch, whose batched
decoder takes fewer waves and more block buffers than the ring decoder: the
records, tile statuses and weights of the two-launch route, with fewer,
about as many and many times more blocks to a workgroup than buffers, with
wave areas sized by the parked output (f32, 16-bit) and by the largest k, and
with failed blocks among them."""
import pytest

import gpu_util as G
from test_gpu_split_layer import Call, general, layer, same

pytestmark = pytest.mark.gpu


def fused(c):
    import haagenti_amd as H
    c.clear()
    tensors = [(r, w, k, o, st) for _, _, r, w, k, o, st in c.tensors]
    rc = c.ctx.hctt_decode_lz4_fused(c.args[0], c.args[0].numel(), c.args[1], c.args[2], c.n, c.st, tensors,
                                     [t["per"] for t in c.L["tensors"]], dtype=c.dt, stream=G.stream())
    assert rc == H.OK
    st, _, out, tst = c.results()
    return [st, out, tst]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("specs,most", [
    ([(1024, 1024, 0.10)], 99),                                     # fewer blocks than workgroups
    ([(4096, 4096, 0.15), (512, 4096, 0.30)], 1),                   # 18 blocks a workgroup, one tile each
    ([(2048, 4096, 0.24), (2048, 4096, 0.05)], 3),                  # as many blocks as buffers, and short ones
    ([(1024, 4096, 0.60), (4096, 2048, 0.12)], 99),                 # coefficient tables above the parks
    ([(1024, 4096, 0.999), (2048, 2048, 0.20)], 2),                 # the largest k
])
def test_against_two_launches(specs, most, dtype):
    c = Call(layer(specs, 7, most=most), dtype)
    st, _, out, tst = general(c)
    assert same(fused(c), [st, out, tst])


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_failed_blocks(dtype):
    L = layer([(2048, 4096, 0.12), (1024, 2048, 0.30)], 8, most=2)
    n = L["in_len"].size
    L["in_len"][[0, 3, 300, 301, n - 1]] = [0, 7, 2, 5, 9]
    L["in_off"][[4, 700]] = 1 << 40
    c = Call(L, dtype)
    st, _, out, tst = general(c)
    assert (tst != 0).sum() >= 7
    assert same(fused(c), [st, out, tst])
