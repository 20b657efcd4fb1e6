"""The tiled attention's splits at their edges: rows and keys around whole
tiles, whole and split blocks, uneven last splits, splits past a row's last
key, several KV heads and head widths, against the oracle's rows; a key that
is infinite is read by the rows that attend it and by no earlier one."""
import math

import numpy as np
import pytest

import oracle as O
from gpu_helpers import empty, spread, to_device, worst_error
from huggingfaceeacp_amd import gemma_q8 as G

pytestmark = pytest.mark.gpu


def attend(torch, q, kc, vc, heads, kvh, hd, rows, offset):
    scale = 1.0 / math.sqrt(hd)
    total = offset + rows
    n = G.mqa_workspace_bytes(rows, heads, hd, total)
    ws = to_device(torch, np.full(n, 0xFF, np.uint8))  # every double a NaN
    out = empty(torch, rows * heads * hd, torch.float32)
    qd, kd, vd = to_device(torch, q), to_device(torch, kc), to_device(torch, vc)
    G.mqa_prefill(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), heads, kvh, hd, rows, offset, scale,
                  out.data_ptr(), ws.data_ptr(), n)
    torch.cuda.synchronize()
    return out.cpu().numpy().reshape(rows, heads * hd), scale


@pytest.mark.parametrize("rows,offset,heads,kvh,hd", [
    (1, 0, 8, 1, 256), (1, 15, 8, 1, 256), (1, 1030, 8, 1, 256), (2, 63, 8, 1, 256),
    (15, 200, 8, 1, 256), (16, 1000, 8, 1, 256), (17, 0, 8, 1, 256), (33, 2015, 8, 1, 256),
    (100, 700, 8, 1, 256), (1, 4130, 2, 1, 64), (9, 500, 4, 2, 128), (40, 900, 6, 2, 64),
    (37, 300, 3, 1, 128), (50, 1100, 16, 1, 128), (20, 4100, 1, 1, 64), (1, 900, 2, 1, 16)])
def test_attention_splits(torch_cuda, rows, offset, heads, kvh, hd):
    total, kw = offset + rows, kvh * hd
    q = spread(rows * heads * hd, 71 + rows, 1.0)
    kc = spread(total * kw, 72, 1.5).astype(np.float16).view(np.uint16)
    vc = spread(total * kw, 73, 1.5).astype(np.float16).view(np.uint16)
    got, scale = attend(torch_cuda, q, kc, vc, heads, kvh, hd, rows, offset)
    for r in sorted({0, 1, rows // 2, rows - 2, rows - 1} & set(range(rows))):
        ref = O.mqa_row_f16(q[r * heads * hd:(r + 1) * heads * hd], kc, vc, heads, kvh, hd,
                            offset + r + 1, scale)
        # both round doubles that differ by sums in another order: one ulp
        assert worst_error(got[r], ref) <= 2.0 ** -23 * 2, f"row {r}"


@pytest.mark.parametrize("rows,offset", [(1, 36), (5, 30), (13, 500)])
def test_an_infinite_value_stays_with_its_rows(torch_cuda, rows, offset):
    """Row r attends keys [0, offset + r]; the last row's value row holds an
    infinity in channel 3.  Earlier rows stay finite, the last row's channel 3
    alone is infinite."""
    heads, kvh, hd, total = 8, 1, 256, offset + rows
    q = spread(rows * heads * hd, 81, 1.0)
    kc = spread(total * hd, 82, 1.0).astype(np.float16).view(np.uint16)
    vc = spread(total * hd, 83, 1.0).astype(np.float16)
    vc[(total - 1) * hd + 3] = np.inf
    got, _ = attend(torch_cuda, q, kc, vc.view(np.uint16), heads, kvh, hd, rows, offset)
    assert np.all(np.isfinite(got[:rows - 1]))
    last = got[rows - 1].reshape(heads, hd)
    assert np.all(np.isposinf(last[:, 3]))
    assert np.all(np.isfinite(np.delete(last, 3, axis=1)))
