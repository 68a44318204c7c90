"""Token ids on their way into the engines: every sequence that int() takes element by element gives the same 32-bit ids, by whichever way it converts."""

import ctypes
from array import array

import numpy as np
import pytest
import torch

from tiny_llm_hip.token_ids import as_int32, token_ids


@pytest.mark.parametrize("tokens", [
    [], (), [5], (1, 2, 3), [True, 0], range(4), b"\x01\x02\x03\x04", bytearray(b"\xff\x00"), [1.0, 2.9], ["7", 8], [2 ** 31, -1, 2 ** 40 + 3],
    [np.int64(4), np.int32(-2)], np.arange(3), np.array([1.5, 2.5]), [torch.tensor(6)], torch.arange(5), array("i", [3, 1]), array("q", [3, 2 ** 33 + 1]), "123",
], ids=lambda t: f"{type(t).__name__}-{len(t)}")
def test_ids_are_those_of_int(tokens):
    flat = [int(t) for t in tokens]
    got = token_ids(tokens)
    assert got.typecode == "i" and list(got) == list((ctypes.c_int32 * len(flat))(*flat))
    assert list(as_int32(got))[:len(flat)] == list(got) and len(as_int32(got)) >= 1


@pytest.mark.parametrize("tokens", [[None], ["x"], [[1]], 5, [float("nan")]])
def test_what_int_refuses_is_refused(tokens):
    with pytest.raises((TypeError, ValueError)):
        token_ids(tokens)
