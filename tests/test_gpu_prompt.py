"""Kernels that prompt-sized steps take, at the edges of their tiles and spans."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hb(bridge):
    import hip_bridge.quant  # noqa: F401

    return bridge


def test_pack_tables_prompt_rows(hb):
    """Rows longer than the workgroup beside empty and one-token rows, first and last too."""
    from hip_bridge import DeviceBuffer

    rng = np.random.default_rng(12)
    row_tokens = np.array([0, 1, 2500, 0, 0, 1023, 1, 1025, 0], np.int32)
    rows, max_pages, page = len(row_tokens), 200, 16
    positions = rng.integers(0, max_pages * page - 2500, rows).astype(np.int32)
    bt = rng.permutation(rows * max_pages).reshape(rows, max_pages).astype(np.int32)
    n = int(row_tokens.sum())
    d = [DeviceBuffer.from_array(a) for a in (row_tokens, positions, bt)]
    out = {k: DeviceBuffer(4 * m) for k, m in (("cu_seqlens", rows + 1), ("token_row", n), ("token_pos", n),
                                              ("kv_slot", n), ("context", rows), ("status", 1))}
    print("case: pack prompt rows", flush=True)
    hb.pack_tables(d[0], d[1], d[2], max_pages, rows, page, *out.values())
    hb.synchronize()
    want = oracle.pack_tables(row_tokens, positions, bt, page)
    assert out["status"].download(np.int32, 1)[0] == 0
    for k in ("cu_seqlens", "token_row", "token_pos", "kv_slot", "context"):
        assert np.array_equal(out[k].download(np.int32, len(want[k])), want[k]), k


# tokens around the 16-token span and the 64-token span group; histories in the
# first span's rows, across its end, in a later span, and past the row's tokens
@pytest.mark.parametrize("in_place", [True, False])
@pytest.mark.parametrize("heads", [(16, 32), (2, 4)])
def test_gdn_prep_spans_equal_the_row_walk(hb, heads, in_place):
    """The span form gives the bits of the form that walks a row (which input
    rows with an odd stride still take): outputs and the rewritten window."""
    from hip_bridge import DeviceBuffer

    hk, hv = heads
    dk, conv, most = 128, 4, 300
    C = 2 * hk * dk + hv * dk
    T = np.array([1, 15, 16, 17, 64, 65, 300, 0, 80, 130], np.int32)
    hist = np.array([0, 300, 16, 14, 20, 64, 17, 5, 80, 62], np.int32)
    rows, n = len(T), int(T.sum())
    rng = np.random.default_rng(hk + in_place)
    bits = lambda *shape: hb.quant.bf16_bits(rng.standard_normal(shape, dtype=np.float32))  # noqa: E731
    slots = rows if in_place else 2 * rows
    win = bits(slots, conv - 1 + most, C)
    src = np.arange(rows, dtype=np.int32)
    dst = src if in_place else src + rows
    wide = np.zeros((n, C + 1), np.uint16)
    wide[:, :C] = bits(n, C)
    ab = bits(n, 2 * hv)
    cu = np.concatenate([[0], np.cumsum(T)]).astype(np.int32)
    conv_w = (rng.standard_normal((C, conv)) * 0.5).astype(np.float32)
    alog, dt = rng.uniform(0, 1, hv).astype(np.float32), rng.standard_normal(hv).astype(np.float32) * 0.1
    got = []
    for ld in (C, C + 1):
        d = [DeviceBuffer.from_array(a) for a in (np.ascontiguousarray(wide[:, :ld]), ab, conv_w, alog, dt, win, hist,
                                                  src, dst, cu)]
        out = [DeviceBuffer(n * w * 4) for w in (hk * dk, hk * dk, hv * dk, hv, hv)]
        print(f"case: gdn prep heads={heads} in_place={in_place} ld={ld}", flush=True)
        hb.call("hb_gdn_prep", d[0], ld, d[1], hb._p(d[1].ptr + 2 * hv), 2 * hv, d[2], d[3], d[4], d[5], d[6], d[7],
                d[8], d[9], rows, hk, hv, dk, dk, conv, most, *out, None)
        hb.synchronize()
        got.append([o.download(np.uint32, n * w) for o, w in zip(out, (hk * dk, hk * dk, hv * dk, hv, hv))]
                   + [d[5].download(np.uint16, win.shape)])
    for name, a, b in zip(("q", "k", "v", "decay", "beta", "window"), *got):
        assert np.array_equal(a, b), f"{name}: {int(np.sum(a != b))} values differ"
