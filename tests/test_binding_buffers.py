"""The address list of a grouped call: lists, tuples and iterators of tensors and of plain addresses,
with None and missing entries as NULL."""
import pytest

import turbo_decode_tail as T


class Buf:
    def __init__(self, p):
        self.p = p

    def data_ptr(self):
        return self.p


ADDRESSES = [4096, 0, 2**47 - 16, 2**63]


@pytest.mark.parametrize("container", [list, tuple, iter, lambda v: (e for e in v)])
@pytest.mark.parametrize("wrap", [lambda a: [Buf(p) for p in a], lambda a: list(a), lambda a: [Buf(a[0]), *a[1:]],
                                  lambda a: [*a[:-1], Buf(a[-1])], lambda a: [a[0], None, *a[2:]]])
def test_addresses_of_any_container(container, wrap):
    assert list(T._ptrs(container(wrap(ADDRESSES)), 4)) == ADDRESSES
    assert list(T._ptrs(container(wrap(ADDRESSES)), 6)) == ADDRESSES + [0, 0]
    with pytest.raises(IndexError):
        T._ptrs(container(wrap(ADDRESSES)), 3)


def test_no_buffers():
    assert list(T._ptrs([], 2)) == [0, 0] and len(T._ptrs((), 0)) == 0
    assert list(T._ptrs([Buf(64)], 0)) == [64]  # beside no matrices one entry is ignored
