"""A batch's encryption in two calls, the messages' encoding between them: the words of the single call; and a refused batch leaves
the next one's random words as they were."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu

CHAINS = {"fp64": [50] * 6 + [50] * 2, "integer": [60] * 6 + [60] * 2, "mixed": [60] + [40] * 5 + [60] * 2}


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,size_p,L,items", [(12, 1, 5, 1), (13, 2, 3, 4), (16, 1, 2, 3)])
def test_two_calls_equal_one(oracle, capi, chain, logn, size_p, L, items):
    cahel, parms, ctx, p = make_pair(oracle, logn, CHAINS[chain], size_p)
    lib, h = capi.lib(), ctx.he_handle()
    rng = np.random.default_rng(logn)
    kp = oracle.chacha_key(3).ctypes.data_as(C.POINTER(C.c_uint32))
    dpk = DeviceArray(capi, host=rand_limbs(p, rng, range(p.size_qp), n_polys=2))
    cts = np.zeros((items, 2, L, p.n), dtype=np.uint64)
    cts[:, 0] = rand_limbs(p, rng, range(L), n_polys=items)
    whole, halves, plains = (DeviceArray(capi, host=x) for x in (cts, np.zeros_like(cts), cts))
    words = lib.he_encrypt_batch_workspace_words(h, L, items)
    ws, other = DeviceArray(capi, shape=(words,)), DeviceArray(capi, shape=(words,))
    capi.check(lib.he_encrypt_begin(h, L, items, dpk.ptr, kp, 11, other.ptr, None))
    capi.check(lib.he_encrypt_batch(h, L, items, dpk.ptr, kp, 11, whole.ptr, ws.ptr, None))
    capi.check(lib.he_memcpy_d2d(halves.ptr, plains.ptr, cts.nbytes, None))
    capi.check(lib.he_encrypt_end(h, L, items, halves.ptr, other.ptr, None))
    assert (halves.numpy() == whole.numpy()).all()
    assert lib.he_encrypt_begin(h, L, 0, dpk.ptr, kp, 11, other.ptr, None) != 0
    assert lib.he_encrypt_begin(h, L, items, None, kp, 11, other.ptr, None) != 0
    assert lib.he_encrypt_end(h, L, items, None, other.ptr, None) != 0
    assert lib.he_encrypt_end(h, 0, items, halves.ptr, other.ptr, None) != 0


def test_a_refused_batch_draws_nothing():
    from lancelot_amd import krum
    a, b = (krum.gpu_init(krum.KrumConfig(log_n=13, seed=5)) for _ in range(2))
    update = np.linspace(-1, 1, 1 << 12).astype(np.float32)
    with pytest.raises(ValueError):
        krum.encrypt_all(a, [np.full(1 << 12, 1e30, np.float32)])
    got, want = krum.encrypt_all(a, [update]), krum.encrypt_all(b, [update])
    assert (got[0][0].to_numpy() == want[0][0].to_numpy()).all()
