"""More than eight special primes: a digit has more limbs than a thread of the fused conversions holds, so every level takes the
conversion kernels limb by limb, and one ciphertext per call.  Everything that switches keys there, against the oracle, with the inner
product inside the blocks pass and as a kernel of its own."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu

CHAINS = {"fp": [50, 49, 48], "int": [60, 58, 55], "mixed": [60, 40, 50]}


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


@pytest.mark.parametrize("separate", ["0", "1"])
@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,size_p,levels", [(9, 9, (18, 10, 2)), (12, 9, (18, 11, 9)), (13, 12, (12, 5)), (16, 10, (3,))])
def test_key_switching(oracle, capi, monkeypatch, logn, size_p, levels, chain, separate):
    """Full and partial last digits, one and two digits, a special limb's block shared by the waves of a workgroup and not."""
    monkeypatch.setenv("CAHEL_HIP_NO_FUSED_KS", separate)
    size_q = -(-levels[0] // size_p) * size_p
    kinds = CHAINS[chain]
    cahel, parms, ctx, p = make_pair(oracle, logn, [kinds[i % 3] for i in range(size_q + size_p)], size_p)
    rng = np.random.default_rng(logn + size_p)
    lib, h, n, K = capi.lib(), ctx.he_handle(), p.n, size_p
    host = [[rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(size_q // K)] for _ in range(2)]
    dev = [[DeviceArray(capi, host=d) for d in key] for key in host]
    evk = [capi.evk_array([d.ptr for d in key]) for key in dev]
    for L in levels:
        beta, tables = -(-L // K), [p.table_index(L, t) for t in range(L + K)]
        ws = DeviceArray(capi, shape=(lib.he_multiply_relin_rescale_workspace_words(h, L),))
        ct, b = (rand_limbs(p, rng, range(L), n_polys=2) for _ in range(2))
        top = np.array(p.moduli[:L], dtype=np.uint64)[:, None] - np.uint64(1)
        ct[1, :, :4] = top
        dct, db, out = DeviceArray(capi, host=ct), DeviceArray(capi, host=b), DeviceArray(capi, shape=(2, L, n))
        y = DeviceArray(capi, shape=(beta, L + K, n))
        capi.check(lib.he_modup(h, L, dct.at(L * n), y.ptr, ws.ptr, None))
        assert (y.numpy() == p.modup(ct[1])).all(), ("modup", L)
        cx = np.stack([rand_limbs(p, rng, tables) for _ in range(2)])
        dcx = DeviceArray(capi, host=cx)
        capi.check(lib.he_moddown(h, L, dcx.ptr, out.ptr, 2, 0, ws.ptr, None))
        assert (out.numpy() == np.stack([p.moddown(x) for x in cx])).all(), ("moddown", L)
        for elt in (0, 5):
            c = p.galois_ntt(ct[1], elt) if elt else ct[1]
            ks = p.key_switch(c, host[0])
            want = np.stack([p.add(b[r], ks[r]) for r in range(2)])
            dout = DeviceArray(capi, host=b)
            capi.check(lib.he_keyswitch(h, L, dct.at(L * n), evk[0], dout.ptr, elt, ws.ptr, None))
            assert (dout.numpy() == want).all(), ("key switch", L, elt)
            dout = DeviceArray(capi, shape=(2, L - 1, n))
            capi.check(lib.he_keyswitch_rescale(h, L, dct.at(L * n), evk[0], db.ptr, dout.ptr, elt, ws.ptr, None))
            assert (dout.numpy() == p.rescale(want)).all(), ("key switch and rescale", L, elt)
        for other, second in ((b, db), (ct, dct)):
            dout = DeviceArray(capi, shape=(2, L - 1, n))
            capi.check(lib.he_multiply_relin_rescale(h, L, dct.ptr, second.ptr, evk[0], dout.ptr, ws.ptr, None))
            assert (dout.numpy() == p.rescale(p.relinearize(p.tensor(ct, other), host[0]))).all(), ("product", L)
        capi.check(lib.he_rotate(h, L, dct.ptr, evk[1], out.ptr, 25, ws.ptr, None))
        assert (out.numpy() == p.apply_galois(ct, 25, host[1])).all(), ("rotation", L)
        elts = [5, 2 * n - 1, 125]
        flat = capi.evk_array([dev[i % 2][d].ptr for i in range(3) for d in range(beta)])
        capi.check(lib.he_hoisted_rotations(h, L, dct.ptr, flat, (C.c_uint32 * 3)(*elts), 3, out.ptr, ws.ptr, None))
        assert (out.numpy() == p.hoisting(ct, elts, [host[i % 2] for i in range(3)])).all(), ("hoisting", L)
        assert (dct.numpy() == ct).all() and (db.numpy() == b).all()
        # batches are refused, not run wrongly
        assert lib.he_multiply_relin_rescale_batch(h, L, 2, dct.ptr, db.ptr, evk[0], out.ptr, ws.ptr, None) == -2


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,size_p,L", [(9, 9, 9), (13, 12, 5)])
def test_encryption(oracle, capi, chain, logn, size_p, L):
    cahel, parms, ctx, p = make_pair(oracle, logn, [CHAINS[chain][i % 3] for i in range(2 * size_p)], size_p)
    rng = np.random.default_rng(logn)
    lib, h, n, Q, K, items = capi.lib(), ctx.he_handle(), p.n, p.size_q, p.size_p, 2
    key = oracle.chacha_key(3)
    pk, plain = rand_limbs(p, rng, range(p.size_qp), n_polys=2), rand_limbs(p, rng, range(L), n_polys=items)
    cts = np.zeros((items, 2, L, n), dtype=np.uint64)
    cts[:, 0] = plain
    dpk, dcts = DeviceArray(capi, host=pk), DeviceArray(capi, host=cts)
    ws = DeviceArray(capi, shape=(lib.he_encrypt_batch_workspace_words(h, L, items),))
    capi.check(lib.he_encrypt_batch(h, L, items, dpk.ptr, key.ctypes.data_as(C.POINTER(C.c_uint32)), 11, dcts.ptr, ws.ptr, None))
    got, tidx = dcts.numpy(), list(range(L)) + list(range(Q, Q + K))
    for k in range(items):
        u = p.ntt_fwd(p.sample_ternary(key, 11 + 3 * k, p.size_qp))
        for i in range(2):
            e = p.ntt_fwd(p.sample_error(key, 12 + 3 * k + i, p.size_qp))
            want = p.moddown(np.ascontiguousarray(p.mul_add(u, pk[i], e)[tidx]))
            assert (got[k, i] == (p.add(want, plain[k]) if i == 0 else want)).all(), (k, i)
