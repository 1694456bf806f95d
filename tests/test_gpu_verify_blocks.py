"""GPU parity of draft rows at 6 and 8 query heads per kv head, whose kernel
takes 4 rows to a page pass in two column blocks (long steps), 2 rows to a
pass (short steps), and one block for segments of up to 2 rows: row counts on
every side of a segment, few and many keys per range, more rows than a
workgroup has threads (256), prompt rows left out, and a workspace that holds
only the 2-row records. Oracle at the bound of tests/_util.close."""
import numpy as np
import pytest
import torch

import pkv
from _util import BS, D, close
from test_gpu_step import i16, i32
from test_gpu_verify import SCALE, run_oracle, run_verify, verify_case

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def default_config():
    pkv.attn_decode_config(1, 32)
    yield
    pkv.attn_decode_config(1, 32)


@pytest.mark.parametrize("G,Hkv,groups", [
    (6, 4, [(40, 4), (7, 3), (1000, 4), (16, 1), (500, 2)]),            # short: halves
    (8, 2, [(33, 4), (129, 5), (64, 6), (1, 4)]),
    (6, 2, [(9000, 4), (7001, 3), (12000, 2), (8000, 5), (3, 4), (6500, 1)]),  # long: whole segments
    (8, 1, [(26000, 4), (15, 7), (3000, 2)]),
    (6, 1, [(int(x), 4) for x in np.random.default_rng(3).integers(1, 900, 70)]),  # more rows than threads
    (8, 4, [(int(x), 1 + i % 4) for i, x in enumerate(np.random.default_rng(4).integers(600, 1500, 30))])])
def test_rows_match_oracle(dev, G, Hkv, groups):
    print(f"case verify blocks G={G} Hkv={Hkv} groups={groups[:6]} ({len(groups)})", flush=True)
    c = verify_case(groups, Hkv, 17 + G, G=G)
    ok, err = close(run_verify(c, dev), run_oracle(c))
    assert ok, f"max |diff| {err}"


@pytest.mark.parametrize("G,Hkv", [(6, 2), (8, 2)])
def test_small_workspace_and_skipped_prompts(dev, G, Hkv):
    """With the bytes of 2 records per row pair the call takes 2-row segments,
    as it did when that was its layout; rows of a prompt (no drafts) are left
    untouched by skip_prompts."""
    print(f"case verify blocks small workspace G={G} Hkv={Hkv}", flush=True)
    groups = [(7000, 4), (300, 3), (9000, 4), (20, 2)]
    c = verify_case(groups, Hkv, 5, G=G)
    T, Hq = c["T"], c["Hq"]
    want = run_oracle(c)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    up = lambda x: (x + 255) // 256 * 256
    rows = (T + cus) * Hq * 2
    small = up(4 * (T + 2)) + up(8 * rows) + 4 * D * rows
    assert small < pkv.attn_verify_workspace(T, Hq)
    args = [i16(c["q"], dev), i16(c["kc"], dev), i16(c["vc"], dev), i16(c["qkv"], dev), c["qstride"], Hq, Hkv]
    args += [i32(c[k], dev) for k in ("pos", "tok_seq", "bt")] + [c["max_blocks"], BS]
    out = torch.full((T, Hq, D), 0x3333, dtype=torch.int16, device=dev)
    ws = torch.empty(small, dtype=torch.uint8, device=dev)
    pkv.attn_verify(*args, out, SCALE, i32(c["cu"], dev), 0, None, 1, T, c["pages"], ws)
    ok, err = close(out.cpu().numpy().view(np.uint16), want)
    assert ok, f"max |diff| {err}"
    outs = np.array([0, -1, 0, 0], np.int32)  # sequence 1 verifies nothing: a prompt
    out.fill_(0x3333)
    ws = torch.empty(pkv.attn_verify_workspace(T, Hq), dtype=torch.uint8, device=dev)
    pkv.attn_verify(*args, out, SCALE, i32(c["cu"], dev), 1, i32(outs, dev), 1, T, c["pages"], ws)
    got = out.cpu().numpy().view(np.uint16)
    skipped = c["tok_seq"] == 1
    assert (got[skipped] == 0x3333).all()
    ok, err = close(got[~skipped], want[~skipped])
    assert ok, f"max |diff| {err}"


@pytest.mark.parametrize("G,Hkv,groups,halves", [
    (6, 4, [(int(x), 4) for x in np.random.default_rng(8).integers(1, 90, 30)], True),      # up to 256 rows
    (6, 2, [(int(x), 4) for x in np.random.default_rng(9).integers(1, 90, 80)], True),      # 320 rows
    (8, 1, [(300, 270), (40, 4), (9, 3), (70, 2)], True),                                   # a long draft run
    (8, 4, [(int(x), 4) for x in np.random.default_rng(10).integers(400, 1000, 70)], False),  # 280 rows, long
    (6, 4, [(9000, 4), (7001, 3), (12000, 2), (8000, 5)], False)])
def test_short_steps_take_half_segments_at_any_row_count(dev, G, Hkv, groups, halves):
    """Under 96 keys a range, segments hold 2 rows, also where the step has more
    rows than the workgroup threads: the word behind the W of the workspace's
    offsets tells the merge."""
    print(f"case verify blocks halves={halves} G={G} Hkv={Hkv} ({len(groups)})", flush=True)
    c = verify_case(groups, Hkv, 23, G=G)
    T, Hq = c["T"], c["Hq"]
    ws = torch.zeros(pkv.attn_verify_workspace(T, Hq), dtype=torch.uint8, device=dev)
    out = torch.zeros(T, Hq, D, dtype=torch.int16, device=dev)
    pkv.attn_verify(i16(c["q"], dev), i16(c["kc"], dev), i16(c["vc"], dev), i16(c["qkv"], dev), c["qstride"], Hq, Hkv,
                    *[i32(c[k], dev) for k in ("pos", "tok_seq", "bt")], c["max_blocks"], BS, out, SCALE,
                    i32(c["cu"], dev), 0, None, 1, T, c["pages"], ws)
    ok, err = close(out.cpu().numpy().view(np.uint16), run_oracle(c))
    assert ok, f"max |diff| {err}"
    assert bool(ws.view(torch.int32)[T + 1].item() & 1 << 30) == halves
