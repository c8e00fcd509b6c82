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


@pytest.mark.parametrize("chain", sorted(CHAINS) + ["two special"])
@pytest.mark.parametrize("logn,L,items,slots,count", [(9, 3, 2, 256, 256), (11, 1, 3, 64, 50), (12, 3, 2, 2048, 2047), (13, 4, 20, 4096, 4096),
                                                      (16, 2, 4, 32768, 32768), (16, 3, 3, 4096, 3000)])
def test_messages_in_moddown(capi, oracle, chain, logn, L, items, slots, count):
    """he_encrypt_end_values against he_ckks_encode_bounded and he_encrypt_end, for messages of both signs up to 2^20 at a scale that
    takes coefficients past every prime, inside ModDown's transform and (12, 3, 2; 16, 2, 4; two special primes) in front of it."""
    bits = CHAINS.get(chain, [60, 40, 40, 40, 50, 50])
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, 1 if chain in CHAINS else 2)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    rng = np.random.default_rng(logn + L)
    kp = oracle.chacha_key(3).ctypes.data_as(C.POINTER(C.c_uint32))
    dpk = DeviceArray(capi, host=rand_limbs(p, rng, range(p.size_qp), n_polys=2))
    values = np.zeros((items, count + 3))
    values[:, :count] = rng.uniform(-1.0, 1.0, (items, count))
    values[0, :] *= 2.0 ** 20
    dvalues = DeviceArray(capi, host=values.view(np.uint64))
    words = lib.he_encrypt_batch_workspace_words(h, L, items)
    ws, encode_ws = DeviceArray(capi, shape=(words,)), DeviceArray(capi, shape=(lib.he_ckks_encode_batch_workspace_words(h, items),))
    want, got = DeviceArray(capi, shape=(items, 2, L, n)), DeviceArray(capi, host=np.full((items, 2, L, n), 5, dtype=np.uint64))
    scale = 2.0 ** 38
    capi.check(lib.he_encrypt_begin(h, L, items, dpk.ptr, kp, 11, ws.ptr, None))
    capi.check(lib.he_ckks_encode_bounded(h, dvalues.ptr, None, count, slots, scale, L, items, count + 3, want.ptr, 2 * L, encode_ws.ptr, None))
    capi.check(lib.he_encrypt_end(h, L, items, want.ptr, ws.ptr, None))
    capi.check(lib.he_encrypt_begin(h, L, items, dpk.ptr, kp, 11, ws.ptr, None))
    capi.check(lib.he_encrypt_end_values(h, L, items, dvalues.ptr, count, slots, scale, count + 3, got.ptr, ws.ptr, encode_ws.ptr, None))
    assert (got.numpy() == want.numpy()).all()
    for bad in ((items, dvalues.ptr, count, slots + 1, scale), (items, dvalues.ptr, slots + 1, slots, scale), (0, dvalues.ptr, count, slots, scale),
                (items, None, count, slots, scale), (items, dvalues.ptr, count, slots, 0.0)):
        assert lib.he_encrypt_end_values(h, L, *bad, count + 3, got.ptr, ws.ptr, encode_ws.ptr, None) != 0, bad
