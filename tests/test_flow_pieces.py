"""The pieces of a large draw cover it in order, start on whole launches and leave no small rest, whose
launches would cost as much as a full piece's."""
import pytest

from pibronic_amd.flow import Flow


@pytest.mark.parametrize("D", [512, 1024])
@pytest.mark.parametrize("B", [128, 65536, 81920, 82048, 98304, 98432, 163968, 196736, 212992, 262144, 1 << 20])
def test_pieces(D, B):
    fl = Flow.__new__(Flow)
    fl.D, fl.num_cu = D, 256
    launch = 128 * fl.num_cu
    pieces = fl._chunks(B)
    assert [p.start for p in pieces[1:]] == [p.stop for p in pieces[:-1]] and (pieces[0].start, pieces[-1].stop) == (0, B)
    assert (len(pieces) == 1) == (4 * B * D <= 320 << 20)
    if len(pieces) > 1:
        assert all(p.start % launch == 0 for p in pieces)
        assert min(p.stop - p.start for p in pieces) > launch // 2
        assert max(4 * D * (p.stop - p.start) for p in pieces) <= 192 << 20
