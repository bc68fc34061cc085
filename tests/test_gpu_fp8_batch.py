"""FP8 projections of nine or more activation rows (whole MFMA tiles) and the
routed experts on the (expert, row) pairs of a prompt chunk, at sizes on the
edges of the row, column and token tiles.

Bars: linear, dual and MLP rows have the bits of one-row calls.  The pairs
are held to the oracle, whose sums run in another order: fp32 sums, fp32
activations and the SiLU intermediate as bf16 hi + lo (at most 2^-17 relative
each), rel-L2 2e-5.
"""

from __future__ import annotations

import subprocess
import sys
import threading

import numpy as np
import pytest
import torch

from conftest import rel_l2
from pocketlm_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nat():
    from pocketlm_amd import native

    assert native.native_fp8_linear_available(), "libpocketlm_hip.so must load on the GPU box"
    return native


def _fp8(rows, cols, seed, nan_at=()):
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn((rows, cols), generator=g) * 0.02).to(torch.float8_e4m3fn).view(torch.uint8)
    for r, c in nan_at:
        w[r, c] = 0x7F
    s = torch.rand(((rows + 127) // 128, (cols + 127) // 128), generator=g) * 9e-3 + 1e-3
    return w.cuda(), s.cuda()


def _x(m, k, seed, dtype):
    return torch.randn((m, k), generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def _rows_of(fn, x, at):
    return torch.cat([fn(x[i:i + 1]) for i in at])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols", [(72, 144), (200, 2064), (576, 7168), (130, 1024), (4200, 144)])
def test_rows_have_the_bits_of_one_row_calls(nat, rows, cols, dtype):
    w, s = _fp8(rows, cols, rows + cols, nan_at=[(rows - 1, 17)])
    w2, s2 = _fp8(rows, cols, rows + cols + 1)
    for m in (9, 16, 17, 33, 64, 65, 129, 150):
        print("linear", rows, cols, m, dtype, flush=True)
        x = _x(m, cols, m, dtype)
        at = sorted({0, 8, 15, 16, m // 2, m - 2, m - 1} & set(range(m)))
        y = nat.fp8_e4m3_block_linear_f32(w, s, x)
        assert torch.isfinite(y).all()
        assert torch.equal(y[at], _rows_of(lambda r: nat.fp8_e4m3_block_linear_f32(w, s, r), x, at)), m
        ya, yb = nat.fp8_e4m3_block_dual_linear_f32(w, s, w2, s2, x)
        assert torch.equal(ya, y) and torch.equal(yb, nat.fp8_e4m3_block_linear_f32(w2, s2, x)), m


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("inter,hid", [(144, 400), (272, 1040), (2048, 512)])
def test_mlp_rows_have_the_bits_of_one_row_calls(nat, inter, hid, dtype):
    args = [*_fp8(inter, hid, 1, nan_at=[(3, 5)]), *_fp8(inter, hid, 2), *_fp8(hid, inter, 3, nan_at=[(hid - 1, 0)])]
    for m in (9, 16, 31, 65, 129, 150):
        print("mlp", inter, hid, m, dtype, flush=True)
        x = _x(m, hid, m, dtype)
        at = sorted({0, 8, 15, 16, m // 2, m - 1} & set(range(m)))
        y = nat.fp8_e4m3_block_mlp_f32(*args, x)
        assert torch.equal(y[at], _rows_of(lambda r: nat.fp8_e4m3_block_mlp_f32(*args, r), x, at)), m


def test_infinite_activation_among_many_rows(nat):
    w, s = _fp8(192, 512, 77)
    x = _x(20, 512, 78, torch.float32)
    x[3, 130] = float("inf")
    x[17, 5] = -float("inf")
    y = nat.fp8_e4m3_block_linear_f32(w, s, x)
    want = _rows_of(lambda r: nat.fp8_e4m3_block_linear_f32(w, s, r), x, range(20))
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.nan_to_num(), want.nan_to_num())
    assert y[3].isinf().any() and torch.isfinite(y[4]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("experts,batch,inter,hid,top", [(3, 9, 144, 400, 1), (70, 40, 128, 272, 4),
                                                         (2, 33, 272, 528, 2), (5, 300, 128, 128, 2)])
def test_pairs_vs_the_oracle(nat, oracle_mod, experts, batch, inter, hid, top, dtype):
    """Experts no row chose, more rows than a tile, duplicate pairs, pairs
    that cancel, zero weights, NaN weight bytes, and pairs out of range."""
    rng = np.random.default_rng(experts + batch)
    items = [(*_fp8(inter, hid, 10 * e, nan_at=[(1, 2)] if e == 1 else ()), *_fp8(inter, hid, 10 * e + 1),
              *_fp8(hid, inter, 10 * e + 2)) for e in range(experts)]
    x = _x(batch, hid, 5, dtype)
    pick = np.stack([rng.choice(max(experts - 1, top), top, replace=False) for _ in range(batch)])
    pi, pr = pick.reshape(-1), np.repeat(np.arange(batch), top)
    pw = rng.uniform(0.1, 1.0, pi.size).astype(np.float32)
    pw[::7] = 0.0
    pi = np.concatenate([pi, pi[:3], pi[3:4]])
    pr = np.concatenate([pr, pr[:3], pr[3:4]])
    pw = np.concatenate([pw, np.float32([0.5, 0.25, 0.125]), -pw[3:4]])
    host = [tuple(t.cpu().numpy() for t in it) for it in items]
    want = oracle_mod.fp8_mlp_many_pair_weighted(host, x.float().cpu().numpy(), pi, pr, pw)
    args = [torch.from_numpy(a).cuda() for a in (pi.astype(np.int64), pr.astype(np.int64), pw)]
    got = nat.fp8_e4m3_block_mlp_many_pair_weighted_f32(items, x, *args)
    assert rel_l2(got.cpu().numpy(), want) < 2e-5
    bad = [torch.cat([a, torch.tensor(v, dtype=a.dtype, device="cuda")])
           for a, v in zip(args, ([experts, -1, 0], [0, 0, batch], [1.0, 1.0, 1.0]))]
    out, n = nat.fp8_e4m3_block_mlp_many_pair_weighted_nosync(items, x, *bad)
    assert int(n.item()) == 3 and torch.equal(out, got)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_other_entry_points_have_the_bits_of_one_row_calls(nat, dtype):
    """Weights of several sizes in one call, 8-row tiles, and the many-expert
    MLPs (66 experts: two tables of addresses), below and above the panel
    kernel's row counts."""
    weights = [_fp8(rows, 400, rows) for rows in (24, 136, 300)]
    packed = [nat.pack_fp8_tiles8(w) for w, _s in weights]
    items = [(*_fp8(48, 144, 3 * e), *_fp8(48, 144, 3 * e + 1), *_fp8(144, 48, 3 * e + 2)) for e in range(66)]
    route = torch.rand((66, 260), generator=torch.Generator().manual_seed(1)).cuda()
    for m in (9, 20, 40, 150, 260):
        print("entry points", m, dtype, flush=True)
        x = _x(m, 400, m, dtype)
        for (w, s), p, y in zip(weights, packed, nat.fp8_e4m3_block_linear_many_f32(weights, x)):
            want = nat.fp8_e4m3_block_linear_f32(w, s, x)
            assert torch.equal(y, want)
            assert torch.equal(nat.fp8_e4m3_block_linear_tiles8_f32(p, s, x), want)
            assert torch.equal(want[m - 1:], nat.fp8_e4m3_block_linear_f32(w, s, x[m - 1:]))
        h = _x(m, 144, m + 1, dtype)
        many = nat.fp8_e4m3_block_mlp_many_f32(items, h)
        for e in (0, 1, 63, 64, 65):
            assert torch.equal(many[e], nat.fp8_e4m3_block_mlp_f32(*items[e], h)), e
        r = route[:, :m].contiguous()
        rows = nat.fp8_e4m3_block_mlp_many_row_weighted_f32(items, h, r)
        for i in (0, 8, m - 1):
            one = nat.fp8_e4m3_block_mlp_many_row_weighted_f32(items, h[i:i + 1], r[:, i:i + 1].contiguous())
            assert torch.equal(rows[i:i + 1], one), i


def _graph_us(calls):
    """Microseconds a call on the device: the calls in a graph, fastest of five replays."""
    graph = torch.cuda.CUDAGraph()
    for call in calls:
        call()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        kept = [call() for call in calls]
    times = []
    for _ in range(6):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        graph.replay()
        end.record()
        torch.cuda.synchronize()
        times.append(start.elapsed_time(end) * 1e3 / len(kept))
    return min(times[1:])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("cols,outs", [(7168, (2048, 2048)), (1024, (512, 512)), (7168, (1536, 576)),
                                       (2048, (1024, 576, 1024)), (7168, (576,)), (7168, (2048,)), (1024, (2048,))])
def test_twelve_rows_take_no_longer_than_eight_and_four(nat, cols, outs, dtype):
    """One call is the faster one (0.4 to 0.8 of the time of two; the bar is
    that it is not the slower one)."""
    sets = [[_fp8(n, cols, 10 * i + j) for j, n in enumerate(outs)] for i in range(8)]
    x = _x(12, cols, 1, dtype)

    def call(weights, rows):
        if len(outs) == 1:
            return nat.fp8_e4m3_block_linear_f32(*weights[0], rows)
        if outs[0] == outs[-1] and len(outs) == 2:
            return nat.fp8_e4m3_block_dual_linear_f32(*weights[0], *weights[1], rows)
        return nat.fp8_e4m3_block_linear_many_f32(weights, rows)

    one = _graph_us([lambda w=w: call(w, x) for w in sets])
    two = _graph_us([lambda w=w: (call(w, x[:8]), call(w, x[8:])) for w in sets])
    print(cols, outs, dtype, one, two, flush=True)
    assert one <= two


# Shapes of the prompt-chunk kernel, LONG rows each: (rows, cols) of a linear,
# (inter, hid) of an MLP.  On 256 compute units they reach every instance of
# it: 64- and 128-row workgroups, K slots together and split, for linear, gate +
# up and down, in both types (tests/test_fp8_plan.py holds them to that); no
# size is a multiple of a tile.
LONG = 509
LONG_LINEARS = [(200, 2064), (8100, 144), (4000, 144), (3100, 272), (1500, 272), (328, 7184)]
LONG_MLPS = [(4048, 272), (1552, 720), (784, 1040), (144, 2064), (144, 4000), (272, 1520)]
LONG_ROWS = (0, 15, 16, 127, 128, 300, 496, 507, 508)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols", LONG_LINEARS)
def test_long_prompt_chunks_have_the_bits_of_one_row_calls(nat, rows, cols, dtype):
    w, s = _fp8(rows, cols, rows, nan_at=[(rows - 1, 17), (0, cols - 1)])
    x = _x(LONG, cols, cols, dtype)
    y = nat.fp8_e4m3_block_linear_f32(w, s, x)
    assert torch.isfinite(y).all()
    assert torch.equal(y[list(LONG_ROWS)], _rows_of(lambda r: nat.fp8_e4m3_block_linear_f32(w, s, r), x, LONG_ROWS))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("inter,hid", LONG_MLPS)
def test_long_prompt_chunks_of_the_mlp_have_the_bits_of_one_row_calls(nat, inter, hid, dtype):
    args = [*_fp8(inter, hid, 1, nan_at=[(inter - 1, 5)]), *_fp8(inter, hid, 2, nan_at=[(3, hid - 1)]),
            *_fp8(hid, inter, 3, nan_at=[(hid - 1, 0)])]
    x = _x(LONG, hid, hid, dtype)
    y = nat.fp8_e4m3_block_mlp_f32(*args, x)
    assert torch.isfinite(y).all()
    assert torch.equal(y[list(LONG_ROWS)], _rows_of(lambda r: nat.fp8_e4m3_block_mlp_f32(*args, r), x, LONG_ROWS))


def test_scratch_of_a_very_long_chunk_is_bounded(nat):
    """A linear and an MLP of 20000 rows (five passes of 4096): scratch as for
    4096 rows (its packed fp32 copy is 4096 x 384 x 4 = 6.3 MB, the MLP's with
    its intermediate 25 MB, in arenas of whole MB that are kept when a larger
    one replaces them), every row with the bits of one-row calls."""
    w, s = _fp8(200, 272, 1)
    mlp = [*_fp8(272, 1040, 2), *_fp8(272, 1040, 3), *_fp8(1040, 272, 4)]
    x, h = _x(20000, 272, 5, torch.float32), _x(20000, 1040, 6, torch.float32)
    at = (0, 4095, 4096, 8191, 8192, 19999)
    box = {}

    def run():
        lib = _lib.load()
        box["linear"] = nat.fp8_e4m3_block_linear_f32(w, s, x)
        box["linear bytes"] = lib.pocketlm_scratch_bytes()
        box["mlp"] = nat.fp8_e4m3_block_mlp_f32(*mlp, h)
        box["mlp bytes"] = lib.pocketlm_scratch_bytes()
        torch.cuda.synchronize()
        lib.pocketlm_release_scratch()

    thread = threading.Thread(target=run)
    thread.start()
    thread.join()
    assert box["linear bytes"] <= 8 << 20 and box["mlp bytes"] <= 48 << 20, box
    assert torch.equal(box["linear"][list(at)], _rows_of(lambda r: nat.fp8_e4m3_block_linear_f32(w, s, r), x, at))
    assert torch.equal(box["mlp"][list(at)], _rows_of(lambda r: nat.fp8_e4m3_block_mlp_f32(*mlp, r), h, at))


def test_prompt_calls_captured_cold():
    """The first panel-kernel calls of a process, made under capture (scratch
    and the large-LDS setting included): every replay, with eager work in
    between, equals the eager call."""
    subprocess.run([sys.executable, __file__], check=True, timeout=110)


def _captured_cold(nat):
    w, s = _fp8(328, 1040, 5)
    mlp = [*_fp8(272, 1040, 6), *_fp8(272, 1040, 7), *_fp8(1040, 272, 8)]
    items = [(*_fp8(144, 1040, 3 * e), *_fp8(144, 1040, 3 * e + 1), *_fp8(1040, 144, 3 * e + 2)) for e in range(5)]
    rows = 300
    x = _x(rows, 1040, 9, torch.float32)
    pi = torch.arange(2 * rows, device="cuda") % 5
    pr = torch.arange(2 * rows, device="cuda") // 2
    pw = torch.rand(2 * rows, generator=torch.Generator().manual_seed(2)).cuda()

    def step():
        return (nat.fp8_e4m3_block_linear_f32(w, s, x), nat.fp8_e4m3_block_mlp_f32(*mlp, x),
                *nat.fp8_e4m3_block_mlp_many_pair_weighted_nosync(items, x, pi, pr, pw))

    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for trial in range(3):
        x.copy_(_x(rows, 1040, 20 + trial, torch.float32))
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in captured]
        for a, b in zip(got, step()):
            assert torch.equal(a, b), trial


if __name__ == "__main__":
    from pocketlm_amd import native

    _captured_cold(native)
