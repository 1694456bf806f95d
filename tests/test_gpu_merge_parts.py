"""GPU parity of the merge of few (row, head) blocks, 64 dims to a block:
record counts below, at and above one round of 256 (4 records to a wave's
load), several tokens, rows with one record (written in place), E4M3 and
draft rows; with FP8 output copies asked for the whole-head merge runs and
gives the same rows within the bound. Oracle at tests/_util.close."""
import numpy as np
import pytest
import torch

import oracle
import pkv
from _util import BS, D, close, decode_case
from test_gpu_decode import run_gpu, run_oracle
from test_gpu_e4m3 import run_decode8
from test_gpu_sweep import e4m3_of
from test_gpu_verify import run_oracle as run_oracle_v, run_verify, verify_case

pytestmark = pytest.mark.gpu
SCALE = 1.0 / 16.0


@pytest.fixture(autouse=True)
def default_config():
    pkv.attn_decode_config(1, 32)
    yield
    pkv.attn_decode_config(1, 32)


@pytest.mark.parametrize("lens,G,Hkv,wg,min_range", [
    ([33], 4, 4, 1, 32), ([97], 4, 4, 1, 32), ([2049], 8, 1, 1, 32), ([4096], 4, 4, 1, 16), ([4097], 6, 4, 1, 16),
    ([9000], 4, 2, 2, 16), ([12000], 1, 4, 3, 16), ([700, 20, 3000, 1], 4, 4, 1, 32), ([5000, 31], 6, 4, 1, 32)])
def test_decode(dev, lens, G, Hkv, wg, min_range):
    print(f"case merge parts lens={lens} G={G} Hkv={Hkv} wg={wg} min_range={min_range}", flush=True)
    pkv.attn_decode_config(wg, min_range)
    c = decode_case(lens, G * Hkv, Hkv, sum(lens))
    want = run_oracle(c, cu=c["cu"])
    got = run_gpu(c, dev, cu=c["cu"])
    ok, err = close(got, want)
    assert ok, f"max |diff| {err}"
    T, K = len(lens), G * Hkv * D
    fq = torch.zeros(T, K, dtype=torch.uint8, device=dev)
    fs = torch.zeros(K // 128, T, device=dev)
    pkv.attn_fp8_next(fq, fs, 1, T)
    ok, err = close(run_gpu(c, dev, cu=c["cu"]), want)
    assert ok and bool((fs > 0).all()), f"with FP8 copies: max |diff| {err}"


@pytest.mark.parametrize("lens,G", [([4097], 4), ([20000], 8), ([300, 5000], 6)])
def test_decode_e4m3(dev, lens, G):
    print(f"case merge parts E4M3 lens={lens} G={G}", flush=True)
    c = decode_case(lens, G * 2, 2, sum(lens))
    k8, v8, ks, vs = e4m3_of(c, np.random.default_rng(1), 0.02)
    want = oracle.attn_decode8(c["q"], k8, v8, ks, vs, c["qkv"], c["qstride"], c["Hq"], 2, c["pos"], c["tok_seq"],
                               c["bt"], c["max_blocks"], BS, SCALE, cu=c["cu"])
    ok, err = close(run_decode8(c, k8, v8, ks, vs, dev), want)
    assert ok, f"max |diff| {err}"


@pytest.mark.parametrize("groups,G", [([(4000, 4)], 4), ([(9000, 2)], 6), ([(1200, 3)], 8)])
def test_verify(dev, groups, G):
    print(f"case merge parts verify groups={groups} G={G}", flush=True)
    c = verify_case(groups, 2, 9, G=G)
    ok, err = close(run_verify(c, dev), run_oracle_v(c))
    assert ok, f"max |diff| {err}"
