"""Which items of a launch the workgroups of csrc/wide.h's kernel take, on the host."""

import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HOOKS = os.path.join(HERE, "_build", "libskyrl_testhooks.so")


@pytest.fixture(scope="module")
def take():
    if not os.path.exists(HOOKS):
        subprocess.run(["make", "-C", os.path.join(HERE, "csrc")], check=True)
    fn = ctypes.CDLL(HOOKS, mode=ctypes.RTLD_LOCAL).skyrl_test_wide_items
    fn.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.POINTER(ctypes.c_int32)]
    return fn


@pytest.mark.parametrize("first", range(1, 2500, 250))
def test_every_half_of_every_item_once(take, first):
    """Up to half as many items as CUs, two workgroups for each, whose launch lasts half an item; then no more than the rounds of whole
    items that an eighth of the CUs takes for an XCD's share of them, the last one a half where there are workgroups for both."""
    for items in range(first, first + 250):
        for launched in (4 * items + 5, items + 37, items):  # routed rows: fewer items than the most there can be
            seen = (ctypes.c_int32 * (2 * items))()
            most = take(launched, items, seen)
            assert most > 0 and list(seen) == [1] * (2 * items), (launched, items)
        if items <= 128:
            assert most == 1, items
        else:
            run = -(-items // 8)
            over = [share % 32 for share in (items // 8, run)]
            assert most == max(2 * (share // 32) + (0 if o == 0 else 1 if o <= 16 else 2) for share, o in zip((items // 8, run), over)), items
