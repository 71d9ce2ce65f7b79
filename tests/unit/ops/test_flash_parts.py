"""How the attention backward's sweeps over the query rows are cut (`ds_flash_bwd_parts` in `csrc/attn/flash_bwd.hip`): the host's side."""
import ctypes

import pytest

from deepspeedsyclsupport_amd.ops import op_builder


@pytest.fixture(scope="module")
def parts():
    op_builder.load("ds_hip_ops")
    return ctypes.CDLL(op_builder.so_path("ds_hip_ops")).ds_flash_bwd_parts


@pytest.mark.parametrize("B,Hq,Hk,S", [(2, 12, 3, 4096), (1, 6, 6, 4191), (1, 32, 32, 768), (1, 24, 24, 791), (2, 6, 6, 1860), (1, 80, 20, 1152), (8, 2, 2, 697)])
def test_equal_sweeps_get_equal_parts(parts, B, Hq, Hk, S):
    """Without a mask all key blocks take as long: a part more for some of them is one more to be added up and makes nothing shorter."""
    assert parts(B, Hq, Hk, S, 0) % -(-S // 256) == 0


@pytest.mark.parametrize("causal", [0, 1])
def test_parts_run_at_once(parts, causal):
    """No more than the chip runs where anything is cut, a part of each sweep at least, and none of fewer than four tiles of the longest sweep."""
    for B in (1, 2, 3, 8):
        for Hk in (1, 2, 5, 16, 40, 300):
            for rep in (1, 4, 71):
                for S in (1, 31, 128, 257, 1000, 2049, 5311, 16384, 65536, 200000):
                    blocks, tiles = -(-S // 256), -(-S // 32)
                    n = parts(B, Hk * rep, Hk, S, causal)
                    assert n == blocks or (n > blocks and B * Hk * n <= 256)
                    assert n <= blocks * max(1, rep * tiles // 4)


@pytest.mark.parametrize("B,Hq,Hk,S,least", [(1, 8, 8, 5311, 32), (1, 5, 5, 8192, 48), (1, 20, 20, 2048, 12), (1, 7, 7, 8192, 32), (1, 24, 24, 2048, 8)])
def test_long_sweeps_are_cut_where_there_is_room(parts, B, Hq, Hk, S, least):
    """All sweeps that are longer than half the first one are in two parts, or, where those would not run at once, none is."""
    assert parts(B, Hq, Hk, S, 1) == least
