"""The bulk readers of lc0_amd.NetworkComputation against a stand-in for the library: no GPU, no network."""
import ctypes as C

import numpy as np
import pytest

from lc0_amd import backend as be


class Library:
    """Answers of a computation of three samples; `bulk` and `nan` change them."""

    def __init__(self, bulk=True, nan=None):
        self.bulk = bulk
        self.values = np.arange(9, dtype=np.float32).reshape(3, 3)
        if nan is not None:
            self.values[nan] = np.nan
        self.probs = np.array([0.25, 0.75, 1.0], np.float32)
        self.offsets = np.array([0, 2, 2, 3], np.int32)

    def lc0mi_comp_batch_size(self, h):
        return 3

    def lc0mi_comp_outputs(self, h, policy, *qdm):
        if not self.bulk:
            return -1
        if policy:
            C.memset(policy, 0, 3 * 1858 * 4)
        for to, row in zip(qdm, self.values):
            C.memmove(to, row.ctypes.data, 12)
        return 0

    def lc0mi_comp_legal_policies(self, h, offsets, probs):
        if not self.bulk:
            return -1
        if offsets:
            C.memmove(offsets, self.offsets.ctypes.data, 16)
        if probs:
            C.memmove(probs, self.probs.ctypes.data, 12)
        return 0

    def lc0mi_comp_legal_policy(self, h, sample, n):
        if not 0 <= sample < 3:
            return None
        n._obj.value = int(self.offsets[sample + 1] - self.offsets[sample])
        return C.cast(self.probs.ctypes.data + 4 * int(self.offsets[sample]), C.POINTER(C.c_float))

    def lc0mi_comp_q(self, h, sample):
        return float("nan")

    lc0mi_comp_d = lc0mi_comp_m = lc0mi_comp_q

    def lc0mi_last_error(self):
        return b"what the library says"


def _computation(lib):
    comp = be.NetworkComputation.__new__(be.NetworkComputation)
    comp._lib, comp._h, comp._values, comp._legal = lib, C.c_void_p(1), None, None
    comp.close = lambda: None
    return comp


def test_results_hands_out_what_the_library_gives():
    got = _computation(Library()).results()
    np.testing.assert_array_equal(np.stack([got["q"], got["d"], got["m"]]), np.arange(9, dtype=np.float32).reshape(3, 3))
    assert got["policy"].shape == (3, 1858)


@pytest.mark.parametrize("which", [0, 1, 2])
def test_nan_is_an_error_in_every_reader(which):
    comp = _computation(Library(nan=(which, 1)))
    with pytest.raises(be.BackendError):
        comp.results()
    reader = (comp.GetQVal, comp.GetDVal, comp.GetMVal)[which]
    assert reader(0) == 3 * which
    with pytest.raises(be.BackendError):
        reader(1)


@pytest.mark.parametrize("bulk", [True, False])
def test_legal_policies_with_and_without_the_bulk_read(bulk):
    comp = _computation(Library(bulk=bulk))
    for sample, want in enumerate(([0.25, 0.75], [], [1.0])):
        got = comp.GetLegalPolicy(sample)
        assert got.dtype == np.float32
        np.testing.assert_array_equal(got, np.array(want, np.float32))
    with pytest.raises(be.BackendError, match="what the library says"):
        comp.GetLegalPolicy(3)
