"""A prefill product over sign tiles is launched with no more parts of K than a row has blocks (no GPU needed: host checks only)."""
import ctypes

import innova_amd as ia


def test_parts_without_blocks_are_refused():
    # oilhip::check_sign_parts(unsigned, unsigned) of common.h
    check = ctypes.CDLL(ia._lib.LIB_PATH)._ZN6oilhip16check_sign_partsEjj
    for bpr in (1, 2, 4, 11, 43):
        for parts in range(0, 17):
            assert (check(bpr, parts) == 0) == (1 <= parts <= bpr), (bpr, parts)
            if 1 <= parts <= bpr:
                bounds = [bpr * p // parts for p in range(parts + 1)]
                assert all(a < b for a, b in zip(bounds, bounds[1:]))        # as the kernel cuts them
