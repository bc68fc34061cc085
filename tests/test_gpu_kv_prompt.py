"""A prompt of more than 8 rows through the dense layer
(kv_dense_layer_prefill_u16_ext_packed_rows8: all rows through each step
together) against the oracle's one row at a time: token counts at the edges
of the token tiles and of the 128-row passes, partial row tiles, K slices,
heads of every kernel variant, over an earlier context with tentative rows.

Bar: rel-L2 1e-3 a row, that of the decode steps' test (the layer's 16-bit
roundings, which a sum in another order can turn the other way).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import kv_dense as kvo
from test_gpu_kv_dense import NAMES, _bits, _device_layer, _layer, _rel, _t

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nat():
    from pocketlm_amd import native

    assert native.native_fp8_linear_available(), "libpocketlm_hip.so must load on the GPU box"
    return native


@pytest.mark.parametrize("dtype,extras,shape,ctx,rows", [
    (torch.float16, False, (256, 512, 8, 2), 30, 9),     # heads of 32
    (torch.bfloat16, True, (256, 512, 8, 2), 0, 16),
    (torch.float16, True, (512, 384, 4, 4), 5, 17),      # heads of 128, no grouping
    (torch.bfloat16, False, (960, 640, 15, 5), 70, 33),  # 3 query heads per kv head
    (torch.float16, False, (896, 1184, 14, 2), 64, 65),  # 7 query heads per kv head, several K slices
    (torch.bfloat16, True, (896, 1184, 14, 2), 200, 129),  # two passes
    (torch.float16, True, (1024, 256, 4, 1), 40, 20),    # heads of 256
    (torch.float16, False, (480, 256, 12, 4), 20, 12),   # heads of 40
    (torch.float16, False, (288, 272, 9, 3), 20, 12),    # 272 columns: one row at a time
])
def test_prompt_rows_match_the_oracle(nat, dtype, extras, shape, ctx, rows):
    H, I, nh, nkv = shape
    dc = 1 if dtype == torch.bfloat16 else 0
    kvw = H // nh * nkv
    w, norms, extra, rng = _layer(H + I + rows, H, I, nh, nkv, dc, extras, scale=0.02)
    dev_w, opt = _device_layer(nat, w, norms, extra, dtype)
    total = ctx + rows + 3
    ours = nat.NativeKvSession(layer_count=2, max_seq_len=total, kv_width=kvw, dtype=dtype)
    ora = kvo.KvSessionOracle(2, total, kvw, dc)
    pre = kvo.f32_to_u16(rng.standard_normal((2, total, kvw)).astype(np.float32), dc)
    if ctx:
        ours.append_committed(1, _t(pre[0][:ctx], dtype), _t(pre[1][:ctx], dtype), count=ctx)
        ora.append(1, pre[0][:ctx], pre[1][:ctx], tentative=False)
    for layer in (0, 1):  # two drafted rows in each layer
        ours.append_tentative(layer, _t(pre[0][ctx:ctx + 2], dtype), _t(pre[1][ctx:ctx + 2], dtype), count=2)
        ora.append(layer, pre[0][ctx:ctx + 2], pre[1][ctx:ctx + 2], tentative=True)
    hidden = kvo.f32_to_u16(rng.standard_normal((rows, H)).astype(np.float32), dc)
    kw = dict(num_heads=nh, num_kv_heads=nkv, rms_eps=1e-6, rope_theta=10000.0)
    got = ours.dense_layer_prefill_packed_rows8(1, _t(hidden, dtype).reshape(rows, H), *dev_w, hidden_size=H,
                                                intermediate_size=I, **kw, **opt)
    got = kvo.u16_to_f32(_bits(got), dc).reshape(rows, H)
    for r in range(rows):
        want = ora.dense_layer_decode(1, hidden[r], norms["in"], norms["post"], *[w[n] for n in NAMES], **kw, **extra)
        ora.commit(1)
        rel = _rel(got[r], kvo.u16_to_f32(want, dc))
        assert rel <= 1e-3, (r, rel)
    for layer in (0, 1):
        assert (ours.committed_length(layer), ours.tentative_length(layer)) == \
            (ora.committed_length(layer), ora.tentative_length(layer))
    for a, b in zip(ours.copy_layer(1), ora.copy_layer(1)):
        af, bf = kvo.u16_to_f32(_bits(a), dc), kvo.u16_to_f32(b, dc)
        close = np.abs(_bits(a).astype(np.int32) - b.astype(np.int32)) <= 1
        assert np.all(close | (np.abs(af - bf) <= 1e-3 * np.abs(bf).max()))
    with pytest.raises(RuntimeError, match="code 4"):
        ours.dense_layer_prefill_packed_rows8(1, _t(hidden, dtype).reshape(rows, H), *dev_w, hidden_size=H,
                                              intermediate_size=I, **kw, **opt)
    ours.close()
