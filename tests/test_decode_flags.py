"""The decode kernel's completion flags share their words with other launches'
partials: a flag is no number that arithmetic leaves behind."""

import ctypes

import numpy as np


def test_flags_are_signalling_nans():
    from toklet_amd import build

    lib = ctypes.CDLL(build.LIB)
    lib.tkh_decode_flag.restype = lib.tkh_decode_epochs.restype = ctypes.c_uint32
    last = lib.tkh_decode_epochs()
    assert last > 1 << 20
    # One past the last is what the bounded-wait hook makes the merge wait for.
    epochs = np.unique(np.concatenate([np.arange(1, 1000), np.geomspace(1, last, 500).astype(np.int64), [last, last + 1]]))
    flags = np.array([lib.tkh_decode_flag(int(e)) for e in epochs], np.uint32)
    assert len(np.unique(flags)) == len(epochs)
    # NaN with a payload, and the bit clear that every arithmetic result's NaN has set.
    assert np.all(np.isnan(flags.view(np.float32))) and np.all(flags & np.uint32(1 << 22) == 0)
