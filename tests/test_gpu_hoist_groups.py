"""Hoisted rotations of batches: how many items a thread serves, and in which order the workgroups run."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


# items a thread at 256 CUs: 2 (576 workgroups of four, below ten for every four CUs), 2 + 1 as 3, 3 + 2, 4 + 3, all of 4, 3 x 3
@pytest.mark.parametrize("unit", [1, 8, 512])
@pytest.mark.parametrize("logn,bits,size_p,L,items", [
    (14, [60, 40, 40, 60], 1, 2, 9), (16, [60, 40, 40, 60], 1, 2, 3), (14, [50] * 8, 2, 5, 5), (14, [60] * 8, 2, 5, 7),
    (16, [60, 40, 40, 60], 1, 2, 4), (15, [60, 40, 40, 60], 1, 2, 9)])
def test_items_of_a_thread(oracle, capi, logn, bits, size_p, L, items, unit):
    """Every item against the call for it alone (another kernel), the last one against the oracle; steps that are gathered from anywhere
    (unit 1), inside stretches of 4,096 words (N / 8192) and inside blocks of 256 words (N / 512)."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, size_p)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    rng = np.random.default_rng(logn + items)
    beta = -(-L // size_p)
    step = 1 if unit == 1 else n // (8192 if unit == 8 else 512)
    elts = [pow(5, step * k, 2 * n) for k in (1, 2, 3)]
    host = [[rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(beta)] for _ in range(2)]
    dev = [[DeviceArray(capi, host=k) for k in key] for key in host]
    flat = capi.evk_array([dev[i % 2][d].ptr for i in range(3) for d in range(beta)])
    d_elts = (C.c_uint32 * 3)(*elts)
    cts = np.stack([rand_limbs(p, rng, range(L), n_polys=2) for _ in range(items)])
    din, dout, one = DeviceArray(capi, host=cts), DeviceArray(capi, shape=cts.shape), DeviceArray(capi, shape=(2, L, n))
    ws = DeviceArray(capi, shape=(lib.he_keyswitch_batch_workspace_words(h, L, items),))
    capi.check(lib.he_hoisted_rotations_batch(h, L, items, din.ptr, flat, d_elts, 3, 0, dout.ptr, ws.ptr, None))
    got = dout.numpy()
    for k in range(items):
        capi.check(lib.he_hoisted_rotations(h, L, din.at(2 * L * n * k), flat, d_elts, 3, one.ptr, ws.ptr, None))
        assert (one.numpy() == got[k]).all(), k
    assert (got[-1] == p.hoisting(cts[-1], elts, [host[i % 2] for i in range(3)])).all()
    capi.check(lib.he_hoisted_rotations_batch(h, L, items, din.ptr, flat, d_elts, 3, 1, dout.ptr, ws.ptr, None))
    added = dout.numpy()
    for k in range(items):
        assert (added[k] == np.stack([p.add(got[k][i], cts[k][i]) for i in range(2)])).all(), k
