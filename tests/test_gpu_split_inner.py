"""Inner products whose blocks are shared by two or four waves, on integers: the waves' 128-bit sums meet before they are reduced, and words
enter them as the last stage leaves them where primes and digits allow it (below 2^60, the waves' sums are cut back from 33 digits on).  Against the oracle, with keys of the
largest residues."""
import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


@pytest.mark.parametrize("logn,bits,size_p,L", [(12, [60] * 5, 1, 4),                # four waves a block, lazy words
                                                 (13, [60] + [40] * 11 + [60] * 4, 4, 10),   # two waves, limbs of both arithmetics
                                                 (12, [60] * 33, 1, 32),              # the last number of digits with lazy words
                                                 (12, [60] * 34, 1, 33),              # the first whose waves' sums could pass 2^128 together
                                                 (12, [60] * 41, 1, 40),
                                                 (12, [60] * 42, 1, 41),
                                                 (12, [60] * 64, 1, 63),              # the most digits of a chain of 64 primes
                                                 (13, [60] * 50, 1, 49),
                                                 (11, [60] * 64, 1, 63)])             # four waves a block
def test_split_inner_products(oracle, capi, logn, bits, size_p, L):
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, size_p)
    rng = np.random.default_rng(L)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    host_evk = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(p.size_q // size_p)]
    for k in host_evk:
        for t in range(p.size_qp):
            k[:, t, : n // 2] = p.moduli[t] - 1
    dev_evk = [DeviceArray(capi, host=k) for k in host_evk]
    ptrs = capi.evk_array([d.ptr for d in dev_evk])
    ws = DeviceArray(capi, shape=(lib.he_keyswitch_workspace_words(h, L),))
    c = rand_limbs(p, rng, range(L))
    c[:, : n // 4] = np.array([p.moduli[t] - 1 for t in range(L)], dtype=np.uint64)[:, None]
    ct = rand_limbs(p, rng, range(L), n_polys=2)
    dc, dct = DeviceArray(capi, host=c), DeviceArray(capi, host=ct)
    dout = DeviceArray(capi, shape=(2, L - 1, n))
    ks = p.key_switch(c, host_evk)
    want = np.stack([p.add(ct[b], ks[b]) for b in range(2)])
    capi.check(lib.he_keyswitch_rescale(h, L, dc.ptr, ptrs, dct.ptr, dout.ptr, 0, ws.ptr, None))
    assert (dout.numpy() == p.rescale(want)).all()
    capi.check(lib.he_keyswitch(h, L, dc.ptr, ptrs, dct.ptr, 0, ws.ptr, None))
    assert (dct.numpy() == want).all()
    drot = DeviceArray(capi, shape=(2, L, n))
    dct = DeviceArray(capi, host=ct)
    capi.check(lib.he_rotate(h, L, dct.ptr, ptrs, drot.ptr, 5, ws.ptr, None))
    ks = p.key_switch(p.galois_ntt(ct[1], 5), host_evk)
    assert (drot.numpy() == np.stack([p.add(p.galois_ntt(ct[0], 5), ks[0]), ks[1]])).all()
