"""GPU tests of the loopback calls that copy between the ranks' tensors directly (no channel count given), at the sizes
where their kernels change course, bit for bit against the oracle's single strided copy."""
import pytest
import torch

from oracle import helix_oracle as ho

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hx():
    import helix_a2a

    assert torch.cuda.is_available()
    return helix_a2a


@pytest.fixture(scope="module")
def ops(hx):
    from helix_a2a import _ops

    return _ops


_WS = {}


def workspace(hx, cp):
    if cp not in _WS:
        _WS.clear()
        _WS[cp] = hx.allocate_workspace(cp, 0)
        for r in range(cp):
            hx.init_workspace(_WS[cp], r, cp)
    return _WS[cp]


def _bits(shape, dtype, offset):
    """Random bits; `offset` elements into an allocation of its own."""
    n = 1
    for d in shape:
        n *= d
    raw = torch.randint(-32768, 32767, (2 * (n + offset),), device="cuda", dtype=torch.int16).view(dtype)
    return raw[offset:offset + n].view(shape)


# (cp, entries, partial_o row elements, statistics row floats, elements the output tensors are shifted by)
CASES = [
    (1, 1, 8, 2, 0),            # one unit, one piece
    (2, 3, 8, 2, 0),
    (3, 1, 504, 6, 0),          # 63 units of a row: the tail of an access
    (3, 5, 512, 6, 0),          # rows of one access
    (3, 5, 520, 6, 0),          # 65 units
    (5, 7, 504, 10, 4),         # rows shorter than an access (four accesses of a pair to a workgroup), outputs 8-byte aligned
    (4, 257, 64, 2, 0),         # whole lines, groups of four accesses, ragged last group
    (7, 33, 1032, 14, 0),       # rows that are no whole lines
    (8, 512, 256, 4, 0),        # 65 536 statistics pieces: the last launch with one piece per thread
    (8, 513, 256, 4, 0),        # ... and the first with four
    (8, 64, 1024, 16, 64),      # whole lines
    (8, 64, 1024, 16, 4),       # ... but outputs that start inside a line
    (32, 9, 128, 8, 0),
    (8, 300, 2048, 16, 0),      # 160 MB in and out: payload past the memory-side cache
    (8, 300, 2056, 16, 0),      # ... with rows that are no whole lines
    (8, 80, 8192, 2, 0),        # ... and few statistics
    (32, 33000, 8, 2, 0),       # more entries than one launch takes
]


@pytest.mark.parametrize("cp,entries,x,s,shift", CASES)
def test_direct_exchange(hx, ops, cp, entries, x, s, shift):
    ws = workspace(hx, cp)
    ins_o = [_bits((entries, cp, x), torch.bfloat16, 0) for _ in range(cp)]
    ins_s = [_bits((entries, cp, s), torch.float32, 0) for _ in range(cp)]
    out = ([_bits((entries, cp, x), torch.bfloat16, shift) for _ in range(cp)],
           [_bits((entries, cp, s), torch.float32, shift // 2) for _ in range(cp)])
    hx.alltoall_loopback(ins_o, ins_s, ws, out=out)
    torch.cuda.synchronize()
    assert ops.device_status() == 0
    for r, want in enumerate(ho.exchange_single_copy([t.view(torch.int16) for t in ins_o])):
        assert torch.equal(out[0][r].view(torch.int16), want), f"partial_o of rank {r}"
    for r, want in enumerate(ho.exchange_single_copy([t.view(torch.int32) for t in ins_s])):
        assert torch.equal(out[1][r].view(torch.int32), want), f"softmax_stats of rank {r}"


def test_direct_and_fifo_exchanges_alternate_on_one_workspace(hx, ops):
    cp = 4
    ws = workspace(hx, cp)
    for i in range(8):
        ins_o = [_bits((19 + i, cp, 128), torch.bfloat16, 0) for _ in range(cp)]
        ins_s = [_bits((19 + i, cp, 4), torch.float32, 0) for _ in range(cp)]
        outs_o, outs_s = hx.alltoall_loopback(ins_o, ins_s, ws, channel_count=(0, 5, 0, 1)[i % 4])
        assert ops.device_status() == 0
        for got, ins, view in ((outs_o, ins_o, torch.int16), (outs_s, ins_s, torch.int32)):
            for r, want in enumerate(ho.exchange_single_copy([t.view(view) for t in ins])):
                assert torch.equal(got[r].view(view), want), (i, r)
