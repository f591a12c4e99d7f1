"""The row transforms and transposes of csrc/dct_fft.hip, which take matrices
with a side above 16384 (the two-pass transforms' limit): every radix of its
FFT, one to four butterflies to a thread, both directions and all output
types; HCT3 fragments scattered in the first pass, by way of a matrix where a
row is too long for that (above 32768), and sides that are no multiples of
512; values at even and odd device addresses; outputs its vector stores can't
take.  (tests/test_host_errors.py checks that these shapes reach it.)

Bound: as in test_gpu_dct_lines.py, a length-N f32 FFT of N / 2 <= 2^14 points
has a relative 2-norm error of about 0.6 eps sqrt(log2 N) from the sums and as
much again from the rounded twiddles, and the real-to-complex step adds two
roundings: below 2e-7 a pass, 3e-7 for two; tested at 1e-6."""
import numpy as np
import pytest

import gpu_util as G
from test_gpu_dct_lines import basis64
from test_gpu_hct3 import H, dec
from test_oracle_hct3 import container, random_fragment

pytestmark = pytest.mark.gpu
REL = 1e-6
# halves of radices 8 and 4 (all), 2 (2048), 3 (192, 24576, 23040), 5 (320,
# 20480, 17920, 23040, 35840), 7 (448, 17920, 28672, 35840)
SHAPES = [(64, 17920), (20480, 192), (23040, 320), (448, 24576), (28672, 128), (2048, 17920), (64, 35840)]
FRAGMENTS = [(512, 17920), (28672, 512), (512, 35840), (320, 17920)]


def rel(got, ref):
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_transforms_vs_f64(rows, cols):
    T, h, c = G.torch(), H(), G.ctx()
    x = T.randn(rows, cols, device="cuda", generator=T.Generator(device="cuda").manual_seed(rows + cols))
    br, bc, xd = basis64(rows), basis64(cols), x.double()
    fwd, inv = T.empty_like(x), T.empty_like(x)
    c.dct_2d(x, rows, cols, fwd, stream=G.stream())
    c.idct_2d(x, rows, cols, inv, stream=G.stream())
    assert rel(fwd, br @ xd @ bc.t().contiguous()) <= REL
    assert rel(inv, br.t().contiguous() @ xd @ bc) <= REL
    for dt, td in ((h.BF16, T.bfloat16), (h.F16, T.float16)):
        out = T.empty(rows, cols, dtype=td, device="cuda")
        c.idct_2d(x, rows, cols, out, dtype=dt, stream=G.stream())
        assert T.equal(out, inv.to(td))


def test_outputs_at_any_element_address():
    # not 16-byte aligned: the dense products, ~1e-6
    T, c = G.torch(), G.ctx()
    rows, cols = SHAPES[0]
    x = T.randn(rows, cols, device="cuda", generator=T.Generator(device="cuda").manual_seed(1))
    want = T.empty_like(x)
    c.idct_2d(x, rows, cols, want, stream=G.stream())
    out = T.full((rows * cols + 2,), 7.0, device="cuda")
    c.idct_2d(x, rows, cols, out.data_ptr() + 4, stream=G.stream())
    assert rel(out[1:-1].view(rows, cols), want.double()) <= 1e-5
    assert float(out[0]) == 7 and float(out[-1]) == 7


@pytest.mark.parametrize("shape", FRAGMENTS)
def test_fragments(shape):
    # three fragments, the second overwriting part of the first, the third
    # running out of values
    T, h = G.torch(), H()
    rng = np.random.default_rng(shape[0])
    total = shape[0] * shape[1]
    bm, v, _ = random_fragment(rng, total, 0.02)
    data = container([random_fragment(rng, total, 0.2), random_fragment(rng, total, 0.05),
                      (bm, v[:v.size // 2], None)])
    coef = dec().reconstruct_coefficients_gpu(data, total, stream=G.stream()).view(*shape).double()
    ref = basis64(shape[0]).t().contiguous() @ coef @ basis64(shape[1])
    got = dec().decompress_to_gpu(data, shape, stream=G.stream()).view(*shape)
    assert rel(got, ref) <= REL
    raw = np.frombuffer(data, np.uint8)
    for odd in (0, 1):
        d_data = G.dev(np.concatenate([np.zeros(odd, np.uint8), raw]))[odd:]
        for dt, td in ((h.F32, T.float32), (h.BF16, T.bfloat16), (h.F16, T.float16)):
            out = T.empty(*shape, dtype=td, device="cuda")
            dec().decompress_device(data, d_data, shape, out, dtype=dt, stream=G.stream())
            assert T.equal(out, got.to(td))
