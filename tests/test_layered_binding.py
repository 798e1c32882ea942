"""LayeredModel.step: what the library is given for the entries that a caller passes, and what is refused before it is asked."""
import ctypes as C
import importlib

import numpy as np
import pytest

layered = importlib.import_module("m40-llm_amd.layered")


class Library:
    def m40host_model_step(self, handle, entries, n, out):
        array = (layered.StepEntryC * n).from_address(entries)
        read = lambda at, count: list((C.c_uint32 * count).from_address(at)) if count else []
        self.got = [(e.sequence_id, read(e.tokens, e.n_tokens), read(e.want, e.n_want)) for e in array]
        return 0


def model():
    m = object.__new__(layered.LayeredModel)
    m.H, m.h, m.vocab = Library(), None, 3
    return m


def test_entries_reach_the_library():
    m = model()
    out = m.step([(np.int64(2), [5, 6, 7], [2, 0, 2]), (True, np.arange(4, dtype=np.int64), []), (0, range(2), (i for i in (1,))), (-1, np.arange(6).reshape(3, 2), np.array([[0], [2]])),
                  (2 ** 32 + 7, (9,), {0: "a"})])
    assert out.shape == (7, 3) and out.dtype == np.float32
    assert m.H.got == [(np.int64(2), [5, 6, 7], [2, 0, 2]), (1, [0, 1, 2, 3], []), (0, [0, 1], [1]), (2 ** 32 - 1, [0, 1, 2], [0, 2]), (7, [9], [0])]


@pytest.mark.parametrize("seq", [1.5, 1.0, "3", None, np.float32(1)])
def test_other_sequence_numbers_are_refused(seq):
    with pytest.raises(TypeError):
        model().step([(0, [1], [0]), (seq, [1], [0])])
