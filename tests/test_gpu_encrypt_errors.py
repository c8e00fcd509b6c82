"""Encryption with one special prime: the errors join ModDown's coefficients, u alone is transformed."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu

CHAINS = {"fp64": [50] * 4 + [50], "integer": [60] * 4 + [60], "mixed": [60] + [40] * 3 + [60], "mixed, small special": [60, 40, 60, 40, 45],
          "small": [30] * 4 + [31]}


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,L,items", [(9, 1, 2), (9, 4, 3), (11, 2, 5), (12, 4, 1), (12, 3, 9), (14, 3, 11), (16, 3, 1), (16, 3, 6)])
def test_errors_in_moddown(oracle, capi, chain, logn, L, items):
    """Both ways into ModDown's transform (behind the special limb's inverse transform, up to 16 limbs of 2^16 words from 2^12 on, and
    inside it), for a random key and for a key of zeros, which leaves the errors alone: a negative one wraps around in the special
    limb and, from there, in every other one."""
    cahel, parms, ctx, p = make_pair(oracle, logn, CHAINS[chain], 1)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    rng = np.random.default_rng(logn + L)
    key, first = oracle.chacha_key(3), 11
    kp = key.ctypes.data_as(C.POINTER(C.c_uint32))
    plain = rand_limbs(p, rng, range(L), n_polys=items)
    cts = np.zeros((items, 2, L, n), dtype=np.uint64)
    cts[:, 0] = plain
    ws = DeviceArray(capi, shape=(lib.he_encrypt_batch_workspace_words(h, L, items),))
    tidx = list(range(L)) + [p.size_q]
    for pk in (rand_limbs(p, rng, range(p.size_qp), n_polys=2), np.zeros((2, p.size_qp, n), dtype=np.uint64)):
        dpk, dcts = DeviceArray(capi, host=pk), DeviceArray(capi, host=cts)
        capi.check(lib.he_encrypt_batch(h, L, items, dpk.ptr, kp, first, dcts.ptr, ws.ptr, None))
        got = dcts.numpy()
        for k in sorted({0, items - 1}):
            u = p.ntt_fwd(p.sample_ternary(key, first + 3 * k, p.size_qp))
            for i in range(2):
                e = p.ntt_fwd(p.sample_error(key, first + 3 * k + 1 + i, p.size_qp))
                want = p.moddown(np.ascontiguousarray(p.mul_add(u, pk[i], e)[tidx]))
                assert (got[k, i] == (p.add(want, plain[k]) if i == 0 else want)).all(), (k, i)
