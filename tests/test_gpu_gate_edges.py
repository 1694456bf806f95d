"""GPU parity of the gated epilogue at its edges: sequences of one key, whose
attention output is that key's V row bit for bit, under gates of 0, +-87.5,
+-88 and -88.5 (where 1 + exp(-gate) lies between 2^126 and the overflow, so
that its reciprocal is denormal and the quotient a small normal or denormal
number), +-89 (where exp overflows), +-100, infinities and NaN, and with
infinite, NaN and the largest V values (G = 4, whose weights are not split into
two bf16 parts). The gated value is within one bf16 ulp of numpy's f32 v / (1 +
exp(-gate)), denormals included: the hardware's exponential is off by up to
2^-16 at these gates (128 in the argument's log2 units, rounded to 24 bits) and
each of the two roundings by half an ulp. NaN, zeros and infinities sit where
numpy has them."""
import numpy as np
import pytest
import torch

from _util import D, bf16_bits, decode_case
from test_gpu_decode import run_gpu
from test_gpu_step import run as run_step, step_case

pytestmark = pytest.mark.gpu
GATES = np.array([np.inf, -np.inf, np.nan, 100, -100, 88.8, -88.8, 0, 3, -3, 1e-3, -20, -87.5, -88, -88.5, 87.5, 88], np.float32)


def f32(bits):
    return (np.ascontiguousarray(bits, np.uint16).astype(np.uint32) << 16).view(np.float32)


@pytest.mark.parametrize("G,entry,special", [(4, "decode", True), (4, "step", True), (6, "step", False),
                                             (8, "decode", False), (2, "decode", False)])
def test_one_key_rows(dev, G, entry, special):
    print(f"case gate edges G={G} {entry}", flush=True)
    lens = [1] * 5
    c = decode_case(lens, G * 4, 4, 3) if entry == "decode" else step_case(lens, 4, 3, 1, G=G)
    T, Hq = len(lens), G * 4
    gates = bf16_bits(np.resize(GATES, D))
    for h in range(Hq):
        c["qkv"][:, h * 512 + 256:h * 512 + 512] = np.roll(gates, h)
    if entry == "decode":
        slot = c["bt"][np.arange(T), 0] * 16
        if special:
            c["vc"][slot[1], 2, :4] = bf16_bits(np.array([np.inf, -np.inf, np.nan, 3e38], np.float32))
        v = c["vc"][slot]
        got = run_gpu(c, dev, cu=c["cu"])
    else:
        if special:
            at = Hq * 512 + 4 * D + 2 * D  # V of kv head 2
            c["qkv"][1, at:at + 4] = bf16_bits(np.array([np.inf, -np.inf, np.nan, 3e38], np.float32))
        v = c["qkv"][:, Hq * 512 + 4 * D:].reshape(T, 4, D)
        got = run_step(c, dev, fused=True)[0]
    g = f32(c["qkv"][:, :Hq * 512].reshape(T, Hq, 2, D)[:, :, 1])
    with np.errstate(all="ignore"):
        want = np.repeat(f32(v), G, axis=1) / (np.float32(1) + np.exp(-g))
    got, want = f32(got).reshape(T, Hq, D), f32(bf16_bits(want))
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    fin = np.isfinite(want)
    assert (np.abs(got - want)[fin] <= np.maximum(np.abs(want[fin]) * 2.0 ** -7, 2.0 ** -133)).all()
