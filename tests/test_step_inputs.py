"""Host arrays of a step as device tensors, and the static decode inputs."""

import numpy as np
import pytest
import torch

from fusioninfer_amd.ops import seqmix
from test_engine import make_engine


@pytest.fixture(scope="module")
def runner():
    return make_engine().runner


def test_to_device_keeps_values_types_and_shapes(runner):
    table = np.arange(6, dtype=np.int64).reshape(2, 3)
    t = runner._to_device({
        "a": ([1, -1, 2 ** 31 - 1], torch.int32),
        "none": ([], torch.long),
        "long": ([2 ** 40, -3], torch.long),
        "table": (table, torch.int32),
        "np": ([np.int64(7)], torch.int32),
    })
    assert t["a"].tolist() == [1, -1, 2 ** 31 - 1]
    assert t["none"].shape == (0,) and t["none"].dtype == torch.long
    assert t["long"].tolist() == [2 ** 40, -3]
    assert t["table"].tolist() == table.tolist()
    assert t["table"].dtype == torch.int32 and t["np"].tolist() == [7]
    for v in t.values():
        assert v.is_contiguous() and v.data_ptr() % 16 == 0


def test_to_device_takes_what_a_tensor_takes(runner):
    """Token ids that a client sent as 7.0, scalars of torch and numpy."""
    for values in ([3, 7.0, True], [torch.tensor(5), 2], [np.int64(4), 1.0],
                   [[1, 2], [3, 4]]):
        t = runner._to_device({"a": (values, torch.long),
                               "b": (values, torch.int32)})
        want = torch.tensor(values, dtype=torch.long)
        assert torch.equal(t["a"], want) and torch.equal(t["b"], want.int())


def test_values_out_of_range_are_refused(runner):
    with pytest.raises(OverflowError):
        runner._to_device({"a": ([2 ** 31], torch.int32)})


@pytest.mark.parametrize("n,bs", [(3, 4), (4, 4), (1, 8)])
def test_decode_inputs_and_padding_rows(runner, n, bs):
    runner._alloc_static(8)
    st = runner._static
    for k, v in st.items():
        v.fill_(5)
    payload = {"ids": list(range(9, 9 + n)), "positions": list(range(n)),
               "slots": [7] * n, "lens": [n + 1] * n,
               "bt": [[3, 2, 1][: i + 1] for i in range(n)][:3] + [[4]] *
               max(0, n - 3)}
    runner._fill_decode_inputs(payload, bs)
    pad = bs - n
    assert st["ids"][:bs].tolist() == payload["ids"] + [0] * pad
    assert st["positions"][:bs].tolist() == payload["positions"] + [0] * pad
    assert st["slots"][:bs].tolist() == payload["slots"] + [-1] * pad
    assert st["seq_lens"][:bs].tolist() == payload["lens"] + [1] * pad
    for i in range(bs):
        own = payload["bt"][i] if i < n else [0]
        assert st["block_tables"][i, : len(own)].tolist() == own
    # ids that are on the device already stay, their padding is cleared
    st["ids"].fill_(6)
    runner._fill_decode_inputs(dict(payload, ids=None), bs)
    assert st["ids"][:bs].tolist() == [6] * n + [0] * pad
    runner._static = {}


@pytest.mark.parametrize("device", ["cpu", pytest.param(
    "cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("window", [0, 24])
def test_context_rows_in_one_copy(device, window):
    """The rows of portions at the start of, within and across blocks, made
    without a wait for the GPU."""
    spans = [(5, 5, [3]), (16, 33, [7, 1, 4]), (1, 50, [9, 2, 8, 0]),
             (40, 40, [5, 6, 10])]
    if device == "cuda":
        torch.cuda.init()
        torch.cuda.set_sync_debug_mode("error")
    try:
        rows = seqmix.ContextRows(spans, 16, device, window)
    finally:
        if device == "cuda":
            torch.cuda.set_sync_debug_mode("default")
    slots, places, first = [], [], 0
    for (n, c, blocks), lo in zip(spans, seqmix.context_starts(spans, window)):
        assert rows.table[len(places), : c - lo].tolist() == list(
            range(first, first + c - lo))
        assert not rows.table[len(places), c - lo:].any()
        slots += [blocks[p // 16] * 16 + p % 16 for p in range(lo, c)]
        places.append(list(range(c - lo - n, c - lo)))
        first += c - lo
    assert rows.count == first and rows.slots.tolist() == slots
    assert rows.positions.tolist() == sum(places, [])
    assert {t.dtype for t in (rows.slots, rows.table, rows.positions)} == {
        torch.int32}
