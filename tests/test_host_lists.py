"""The native readers of ragged Python lists against numpy's element by element walk, over what they take
themselves (exact lists of exact numbers), what they leave to that walk, and what nothing takes."""

import os

import numpy as np
import pytest
import torch

from open_instruct_amd import rl_utils

BIG = 2**63 - 1
INTS = [
    [[1, 2, 3], [], [0, -7, BIG, -BIG - 1]],
    [[], [], []],
    [[True, False], [5]],
    [np.arange(4), [1, 2]],  # left to the walk
    [(1, 0), [2]],
    ([1, 0], [0, 0, 0]),
    [list(range(300)), [0] * 17],
]


@pytest.mark.parametrize("seqs", INTS)
@pytest.mark.parametrize("skip", [0, 2, BIG, 2**64, 0.0, None])
def test_integers(seqs, skip):
    offsets = rl_utils._offsets(seqs)
    assert offsets.tolist() == [0] + np.cumsum([len(s) for s in seqs]).tolist()
    out = np.full(offsets[-1], 77, dtype=np.int64)
    others = rl_utils._fill_ints(seqs, offsets, out, skip)
    assert out.tolist() == [int(x) for s in seqs for x in s]
    assert others.tolist() == [sum(int(x) != skip for x in s) for s in seqs]
    flags = np.full(offsets[-1], 77, dtype=np.uint8)
    rl_utils._fill_flags(seqs, offsets, flags)
    assert flags.tolist() == [int(x != 0) for s in seqs for x in s]


@pytest.mark.parametrize(
    "seqs", [[[-0.5, 1e-45, 3.4e38], [], [float("nan"), float("inf"), 0.1]], [[1, 2.5]], [np.array([0.25], np.float32)], [[]]]
)
def test_floats(seqs):
    offsets = rl_utils._offsets(seqs)
    out = np.full(offsets[-1], 7, dtype=np.float32)
    rl_utils._fill_floats(seqs, offsets, out)
    np.testing.assert_array_equal(out, np.array([x for s in seqs for x in s], dtype=np.float32))


@pytest.mark.parametrize("bad,error", [([["a"]], ValueError), ([[2**63]], OverflowError), ([[None]], TypeError), ([3], TypeError)])
def test_refused(bad, error):
    with pytest.raises(error):
        offsets = rl_utils._offsets(bad)
        rl_utils._fill_ints(bad, offsets, np.empty(offsets[-1], dtype=np.int64), 0)


def test_without_the_native_reader_every_list_takes_the_walk(monkeypatch, tmp_path):
    with_reader = [(rl_utils._offsets(s).tolist(), s) for s in INTS]
    monkeypatch.setattr(rl_utils._lib, "PYLISTS_PATH", str(tmp_path / "none.so"))
    monkeypatch.setattr(rl_utils._lib, "_pylists", None)
    with pytest.warns(RuntimeWarning, match="missing") as caught:
        for expected, seqs in with_reader:
            offsets = rl_utils._offsets(seqs)
            assert offsets.tolist() == expected
            out, flags = np.empty(offsets[-1], dtype=np.int64), np.empty(offsets[-1], dtype=np.uint8)
            others = rl_utils._fill_ints(seqs, offsets, out, 0)
            rl_utils._fill_flags(seqs, offsets, flags)
            assert out.tolist() == [int(x) for s in seqs for x in s] and flags.tolist() == [int(x != 0) for x in out]
            assert others.tolist() == [sum(int(x) != 0 for x in s) for s in seqs]
        floats = np.empty(2, dtype=np.float32)
        rl_utils._fill_floats([[0.5], [2.0]], np.array([0, 1, 2]), floats)
        assert floats.tolist() == [0.5, 2.0]
    assert len(caught) == 1  # one warning, not one per call


def test_the_reader_is_named_after_the_interpreter_it_was_built_for():
    import sysconfig

    assert os.path.basename(rl_utils._lib.PYLISTS_PATH) == "liboi_pylists" + sysconfig.get_config_var("EXT_SUFFIX")
    assert rl_utils._lib.pylists() is not None


def test_a_list_that_changed_since_its_length_was_taken():
    seqs = [[1, 2], [3]]
    offsets = rl_utils._offsets(seqs)
    seqs[1].append(4)
    lib = rl_utils._lib.pylists()
    out, others = np.empty(3, dtype=np.int64), np.empty(2, dtype=np.int64)
    assert lib.oi_py_flatten_ints(seqs, 2, offsets.ctypes.data, 0, out.ctypes.data, others.ctypes.data) == -1


def test_packing_is_refused_while_a_stream_captures(monkeypatch):
    # its inputs are read from host lists: a graph would replay the copy of a buffer that is no longer theirs
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError, match="captured"):
        rl_utils.pack_sequences([[1, 2]], [[3]], [[1]], 8, 0, [[-0.5]], device="cuda")
