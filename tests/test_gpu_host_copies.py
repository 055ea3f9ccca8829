"""Copies of the host-pointer entry points through pinned slots (csrc/zq3d_hostcopy.h): calls of a few bytes, of
just under, at and over a slot (2 MiB) and of many slots, arrays that do not start or end on a slot, the slots
given back in between, and several threads calling at once; every value arrives."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def regular(u, v, w):
    """mac_to_regular4's cell averages, in float as the kernel takes them."""
    h = np.float32(0.5)
    out = np.zeros(u.shape[:2] + (u.shape[2] - 1, 4), np.float32)
    out[..., 0] = h * (u[:, :, :-1] + u[:, :, 1:])
    out[..., 1] = h * (v[:, :-1] + v[:, 1:])
    out[..., 2] = h * (w[:-1] + w[1:])
    return out


def check(W, H, D, seed):
    import zq_smokesimulation_amd as z
    rng = np.random.default_rng(seed)
    u = rng.standard_normal((D, H, W + 1), np.float32)
    v = rng.standard_normal((D, H + 1, W), np.float32)
    w = rng.standard_normal((D + 1, H, W), np.float32)
    got = z.stages.mac_to_regular4(u, v, w)
    assert np.array_equal(got.view(np.uint32), regular(u, v, w).view(np.uint32)), (W, H, D)


# total bytes in and out: some hundred, one slot less a little, a little more, two to thirty slots
@pytest.mark.parametrize("dims", [(3, 2, 2), (55, 56, 55), (56, 56, 56), (64, 64, 32), (64, 64, 33), (101, 83, 71),
                                  (128, 128, 128)])
def test_every_value_arrives(dims):
    from zq_smokesimulation_amd import _lib
    print("copies", dims, flush=True)
    check(*dims, 5)
    _lib.lib().zq3d_release_workspace()
    check(*dims, 6)
    check(*dims, 7)


def test_calls_from_several_threads():
    errors = []

    def work(n):
        try:
            for r in range(3):
                check(40 + 9 * n, 64, 60, 100 * n + r)
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(n,)) for n in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
