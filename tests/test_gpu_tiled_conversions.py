"""Fused base conversions whose inputs the inverse rows pass leaves in the conversion's own order (N = 2^16, from 10 limbs of Ql u P on, 12 on
FP64) against the oracle, on every back end, on both sides of the line, with partial last digits, with scratch that is too small for the
order (the merged ModDown + rescale of one digit), and where data limbs and conversion run on different arithmetic."""
import ctypes

import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu

CASES = [  # bits, size_p, levels
    ([50] * 12 + [50] * 4, 4, (10, 8, 7)),            # FP64: 14 (half a digit), 12 and 11 limbs (natural order)
    ([50] * 8 + [50] * 8, 8, (8, 6)),                 # one digit: scratch for ModDown's inputs but not for the merged one's, and for neither
    ([60] + [40] * 7 + [60] * 4, 4, (8, 6, 5)),       # integer conversion, limbs of both arithmetics; 5: natural order
    ([60] * 8 + [60] * 2, 2, (8, 7)),                 # integers throughout: 10 limbs, and 9
    ([45] * 8 + [60] * 4, 4, (7,)),                   # inverse transform of the data limbs on FP64 in front of an integer conversion
]


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


@pytest.mark.parametrize("bits,size_p,levels", CASES)
def test_key_switches_with_tiled_conversions(oracle, capi, bits, size_p, levels):
    cahel, parms, ctx, p = make_pair(oracle, 16, bits, size_p)
    rng = np.random.default_rng(7)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    host_evk = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(p.size_q // size_p)]
    dev_evk = [DeviceArray(capi, host=k) for k in host_evk]
    ptrs = capi.evk_array([d.ptr for d in dev_evk])
    for L in levels:
        ws = DeviceArray(capi, shape=(lib.he_keyswitch_workspace_words(h, L),))
        c = rand_limbs(p, rng, range(L))
        c[0, :4] = [0, 1, p.moduli[0] - 1, p.moduli[0] - 2]
        ct = rand_limbs(p, rng, range(L), n_polys=2)
        ks = p.key_switch(c, host_evk)
        want = np.stack([p.add(ct[b], ks[b]) for b in range(2)])
        dc, dct = DeviceArray(capi, host=c), DeviceArray(capi, host=ct)
        dout = DeviceArray(capi, shape=(2, L - 1, n))
        capi.check(lib.he_keyswitch_rescale(h, L, dc.ptr, ptrs, dct.ptr, dout.ptr, 0, ws.ptr, None))
        assert (dout.numpy() == p.rescale(want)).all(), L
        capi.check(lib.he_keyswitch(h, L, dc.ptr, ptrs, dct.ptr, 0, ws.ptr, None))
        assert (dct.numpy() == want).all(), L
        # a rotation, and a hoisted one: the automorphism before and after ModUp
        elt = 5
        dct = DeviceArray(capi, host=ct)
        drot = DeviceArray(capi, shape=(2, L, n))
        capi.check(lib.he_rotate(h, L, dct.ptr, ptrs, drot.ptr, elt, ws.ptr, None))
        ks = p.key_switch(p.galois_ntt(ct[1], elt), host_evk)
        assert (drot.numpy() == np.stack([p.add(p.galois_ntt(ct[0], elt), ks[0]), ks[1]])).all(), L
        capi.check(lib.he_hoisted_rotations(h, L, dct.ptr, ptrs, (ctypes.c_uint32 * 1)(elt), 1, drot.ptr, ws.ptr, None))
        cx = p.inner_prod(p.galois_ntt(p.modup(ct[1]), elt), host_evk)
        md = [p.moddown(cx[b]) for b in range(2)]
        assert (drot.numpy() == np.stack([p.add(p.galois_ntt(ct[0], elt), md[0]), md[1]])).all(), L


@pytest.mark.parametrize("bits", [[60] * 8 + [60] * 2, [60] + [40] * 7 + [60] * 2])
def test_batch_of_merged_moddown_with_tiled_conversion(oracle, capi, bits):
    """Three key switches with rescale in one call, conversions in integers: ModDown's inputs lie at the strides of the tiled order, K + 1
    limbs a polynomial, two polynomials an item."""
    L, size_p, items = 8, 2, 3
    cahel, parms, ctx, p = make_pair(oracle, 16, bits, size_p)
    rng = np.random.default_rng(5)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    # the order is taken: limbs in all, and its inputs within what is left of the digits
    assert L + size_p >= 10 and (L + size_p) * items <= 64 and 2 * items * (size_p + 1) <= items * (L // size_p) * (L + size_p)
    host_evk = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(L // size_p)]
    dev_evk = [DeviceArray(capi, host=k) for k in host_evk]
    c = rand_limbs(p, rng, range(L), n_polys=items)
    ct = np.stack([rand_limbs(p, rng, range(L), n_polys=2) for _ in range(items)])
    dc, dct = DeviceArray(capi, host=c), DeviceArray(capi, host=ct)
    ws = DeviceArray(capi, shape=(lib.he_keyswitch_batch_workspace_words(h, L, items),))
    out = DeviceArray(capi, shape=(items, 2, L - 1, n))
    capi.check(lib.he_keyswitch_rescale_batch(h, L, items, dc.ptr, L, capi.evk_array([d.ptr for d in dev_evk]), dct.ptr, out.ptr, 0, ws.ptr,
                                              None))
    got = out.numpy()
    for k in range(items):
        ks = p.key_switch(c[k], host_evk)
        assert (got[k] == p.rescale(np.stack([p.add(ct[k][r], ks[r]) for r in range(2)]))).all(), k


@pytest.mark.parametrize("bits,size_p,L", [([50] * 12, 2, 10), ([60] + [40] * 7 + [60] * 2, 2, 8), ([50] * 16, 8, 4)])
def test_encryption_with_tiled_conversion(oracle, capi, bits, size_p, L):
    """ModDown's inputs lie where the encrypted u was, or in natural order where that is too short (L < K)."""
    cahel, parms, ctx, p = make_pair(oracle, 16, bits, size_p)
    rng = np.random.default_rng(3)
    lib, h, n, Q, K, items = capi.lib(), ctx.he_handle(), p.n, p.size_q, p.size_p, 2
    key = oracle.chacha_key(3)
    pk, plain = rand_limbs(p, rng, range(p.size_qp), n_polys=2), rand_limbs(p, rng, range(L), n_polys=items)
    cts = np.zeros((items, 2, L, n), dtype=np.uint64)
    cts[:, 0] = plain
    dpk, dcts = DeviceArray(capi, host=pk), DeviceArray(capi, host=cts)
    ws = DeviceArray(capi, shape=(lib.he_encrypt_batch_workspace_words(h, L, items),))
    capi.check(lib.he_encrypt_batch(h, L, items, dpk.ptr, key.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), 11, dcts.ptr, ws.ptr, None))
    got, tidx = dcts.numpy(), list(range(L)) + list(range(Q, Q + K))
    for k in range(items):
        u = p.ntt_fwd(p.sample_ternary(key, 11 + 3 * k, p.size_qp))
        for i in range(2):
            e = p.ntt_fwd(p.sample_error(key, 12 + 3 * k + i, p.size_qp))
            want = p.moddown(np.ascontiguousarray(p.mul_add(u, pk[i], e)[tidx]))
            assert (got[k, i] == (p.add(want, plain[k]) if i == 0 else want)).all(), (k, i)
