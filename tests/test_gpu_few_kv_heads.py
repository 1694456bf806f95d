"""GPU parity of decode, verify and the fused step with 1 or 2 kv heads from
the token count on at which a workgroup takes several key ranges (4 waves,
4 / Hkv ranges): token counts below, at and above the block's 256 threads,
ranges shorter and longer than the least kept, sequences of one key, rows of
prompts left out, against the oracle at the bound of tests/_util.close."""
import numpy as np
import pytest
import torch

import oracle
import pkv
from _util import BS, close, decode_case
from test_gpu_decode import run_gpu, run_oracle
from test_gpu_e4m3 import run_decode8
from test_gpu_step import oracle_step, run as run_step, step_case
from test_gpu_sweep import e4m3_of
from test_gpu_verify import run_oracle as run_oracle_v, run_verify, verify_case

pytestmark = pytest.mark.gpu
SCALE = 1.0 / 16.0


@pytest.fixture(autouse=True)
def default_config():
    pkv.attn_decode_config(1, 32)
    yield
    pkv.attn_decode_config(1, 32)


def lens_of(T, hi, seed):
    rng = np.random.default_rng(seed)
    lens = [int(x) for x in rng.integers(1, hi, T)]
    lens[0], lens[T // 2], lens[-1] = 1, 16 * (hi // 16), hi
    return lens


@pytest.mark.parametrize("G,Hkv,T,hi,min_range", [
    (4, 2, 64, 900, 32), (4, 1, 64, 1700, 32), (4, 2, 256, 300, 32), (4, 1, 257, 260, 16), (4, 2, 300, 40, 32),
    (6, 2, 70, 1200, 32), (8, 2, 64, 1500, 32), (8, 1, 66, 1300, 32), (1, 1, 64, 600, 32), (2, 2, 65, 700, 1 << 20)])
def test_decode_and_step(dev, G, Hkv, T, hi, min_range):
    print(f"case few kv heads G={G} Hkv={Hkv} T={T} hi={hi} min_range={min_range}", flush=True)
    pkv.attn_decode_config(1, min_range)
    lens = lens_of(T, hi, T + G)
    c = decode_case(lens, G * Hkv, Hkv, T)
    ok, err = close(run_gpu(c, dev, cu=c["cu"]), run_oracle(c, cu=c["cu"]))
    assert ok, f"decode: max |diff| {err}"
    c = step_case(lens, Hkv, T + 1, 1, G=G)
    got, kc, vc = run_step(c, dev, fused=True)
    plain, _, _ = run_step(c, dev, fused=False)
    want, wkc, wvc = oracle_step(c)
    assert np.array_equal(kc, wkc) and np.array_equal(vc, wvc), "appended rows differ"
    assert np.array_equal(got, plain), "the fused step differs from append + decode"
    ok, err = close(got, want)
    assert ok, f"step: max |diff| {err}"


@pytest.mark.parametrize("G,Hkv,T,hi", [(4, 1, 64, 1500), (4, 2, 128, 1200), (8, 2, 130, 900), (6, 1, 65, 700),
                                        (2, 1, 260, 200)])
def test_decode_e4m3(dev, G, Hkv, T, hi):
    print(f"case few kv heads E4M3 G={G} Hkv={Hkv} T={T} hi={hi}", flush=True)
    c = decode_case(lens_of(T, hi, T), G * Hkv, Hkv, T)
    k8, v8, ks, vs = e4m3_of(c, np.random.default_rng(T), 0.02)
    got = run_decode8(c, k8, v8, ks, vs, dev)
    want = oracle.attn_decode8(c["q"], k8, v8, ks, vs, c["qkv"], c["qstride"], c["Hq"], Hkv, c["pos"], c["tok_seq"],
                               c["bt"], c["max_blocks"], BS, SCALE, cu=c["cu"])
    ok, err = close(got, want)
    assert ok, f"max |diff| {err}"


@pytest.mark.parametrize("G,Hkv,seqs,rows,hi,f8", [(4, 1, 16, 4, 2500, False), (8, 1, 22, 3, 1500, False),
                                                   (4, 1, 22, 3, 1300, True), (8, 1, 17, 4, 1100, True),
                                                   (4, 2, 40, 4, 300, False), (8, 2, 40, 4, 300, True)])
def test_verify(dev, G, Hkv, seqs, rows, hi, f8):
    print(f"case few kv heads verify G={G} Hkv={Hkv} seqs={seqs} rows={rows} hi={hi} f8={f8}", flush=True)
    c = verify_case([(L, rows) for L in lens_of(seqs, hi, seqs)], Hkv, seqs, G=G)
    if f8:
        k8, v8, ks, vs = e4m3_of(c, np.random.default_rng(seqs), 0.02)
        got = run_decode8(c, k8, v8, ks, vs, dev, entry="verify")
        want = oracle.attn_decode8(c["q"], k8, v8, ks, vs, c["qkv"], c["qstride"], c["Hq"], Hkv, c["pos"],
                                   c["tok_seq"], c["bt"], c["max_blocks"], BS, SCALE, cu=c["cu"])
    else:
        got, want = run_verify(c, dev), run_oracle_v(c)
    ok, err = close(got, want)
    assert ok, f"max |diff| {err}"


@pytest.mark.parametrize("G,Hkv,T", [(8, 1, 64), (4, 1, 300)])
def test_noalloc_step(dev, G, Hkv, T):
    """The no-allocation array holds the several-range records of the second
    case only; the first falls back to one range per workgroup."""
    from test_zz_no_alloc import run_step as run_noalloc
    print(f"case few kv heads noalloc G={G} Hkv={Hkv} T={T}", flush=True)
    c = step_case(lens_of(T, 700, T), Hkv, T, 1, G=G)
    got, kc, vc = run_noalloc(c, dev, noalloc=True)
    want, wkc, wvc = oracle_step(c)
    assert np.array_equal(kc, wkc) and np.array_equal(vc, wvc), "appended rows differ"
    ok, err = close(got, want)
    assert ok, f"max |diff| {err}"


@pytest.mark.parametrize("G,Hkv,f8,prompt,rows,multi", [
    (4, 2, True, 200, 100, False), (8, 2, True, 300, 127, False), (4, 2, True, 30, 128, True), (4, 1, True, 33, 70, True),
    (4, 2, False, 200, 40, True), (8, 1, False, 90, 40, True)])
def test_rows_that_attend_choose_the_ranges(dev, G, Hkv, f8, prompt, rows, multi):
    """Over E4M3 at 2 kv heads a prompt left out by skip_prompts doesn't count
    as rows that give a workgroup's several ranges work: the keys per range (the
    word behind the offsets' last, W) are those of one range per workgroup."""
    print(f"case few kv heads mixed G={G} Hkv={Hkv} f8={f8} prompt={prompt} rows={rows}", flush=True)
    lens = [int(x) for x in np.random.default_rng(rows).integers(1000, 3000, rows)]
    c = verify_case([(40, prompt)] + [(L, 1) for L in lens], Hkv, rows, G=G)
    T, Hq = c["T"], c["Hq"]
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    bf = lambda k: t(c[k].view(np.int16))
    meta = [t(c[k]) for k in ("pos", "tok_seq", "bt")]
    out = torch.full((T, Hq, 256), 0x3333, dtype=torch.int16, device=dev)
    ws = torch.zeros(pkv.attn_decode_workspace(T, Hq), dtype=torch.uint8, device=dev)
    tail = [c["max_blocks"], BS, out, SCALE, t(c["cu"]), 1, None, 1, T, c["pages"], ws]
    args = (c["qkv"], c["qstride"], Hq, Hkv, c["pos"], c["tok_seq"], c["bt"], c["max_blocks"], BS, SCALE)
    if f8:
        k8, v8, ks, vs = e4m3_of(c, np.random.default_rng(rows), 0.02)
        pkv.attn_decode_e4m3(bf("q"), t(k8), t(v8), t(ks), t(vs), bf("qkv"), c["qstride"], Hq, Hkv, *meta, *tail)
        want = oracle.attn_decode8(c["q"], k8, v8, ks, vs, *args, cu=c["cu"])
    else:
        pkv.attn_decode(bf("q"), bf("kc"), bf("vc"), bf("qkv"), c["qstride"], Hq, Hkv, *meta, *tail)
        want = run_oracle_v(c)
    got = out.cpu().numpy().view(np.uint16)
    assert (got[:prompt] == 0x3333).all()
    ok, err = close(got[prompt:], want[prompt:])
    assert ok, f"max |diff| {err}"
    W, R = ws.view(torch.int32)[T:T + 2].tolist()
    assert W == sum(lens) + rows
    nb = torch.cuda.get_device_properties(0).multi_processor_count * (2 if f8 else 1)
    per_wg = -(-W // nb)
    assert R == (max(32, -(-W // (nb * 4 // Hkv)), min(128, per_wg)) if multi else max(32, per_wg))
