"""Key switches whose words come near the size of the last-level cache (from 400 limbs of 2^16 words on), where the key's words pass by the
caches, and, in a product, the digits' words as well: on chains with limbs of both arithmetics, with the key's pointers among the kernel's
arguments (three digits) and in its table (more), against the oracle."""
import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


@pytest.mark.parametrize("bits,size_p,L", [([60] + [40] * 23 + [60] * 8, 8, 24),     # three digits: 448 limbs in all
                                            ([60] + [40] * 17 + [60] * 3, 3, 16),     # five digits and a limb: 444
                                            ([60] + [40] * 10 + [60], 1, 11),         # the most digits that work their twiddles out: 464
                                            ([60] + [40] * 11 + [60], 1, 12)])        # the first that read them: 542
def test_key_words_past_the_caches_on_mixed_chains(oracle, capi, bits, size_p, L):
    cahel, parms, ctx, p = make_pair(oracle, 16, bits, size_p)
    lib, h, n, beta = capi.lib(), ctx.he_handle(), p.n, -(-L // size_p)
    assert (3 * beta + 2) * (L + size_p) + 4 * L >= 400
    rng = np.random.default_rng(L)
    host_evk = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(beta)]
    dev_evk = [DeviceArray(capi, host=k) for k in host_evk]
    ptrs = capi.evk_array([d.ptr for d in dev_evk])
    a, b = (rand_limbs(p, rng, range(L), n_polys=2) for _ in range(2))
    da, db = DeviceArray(capi, host=a), DeviceArray(capi, host=b)
    ws = DeviceArray(capi, shape=(lib.he_multiply_relin_rescale_workspace_words(h, L),))
    # keys alone
    ks = p.key_switch(b[1], host_evk)
    want = np.stack([p.add(a[r], ks[r]) for r in range(2)])
    dct = DeviceArray(capi, host=a)
    capi.check(lib.he_keyswitch(h, L, db.at(L * n), ptrs, dct.ptr, 0, ws.ptr, None))
    assert (dct.numpy() == want).all()
    elt = pow(5, 3, 2 * n)
    drot = DeviceArray(capi, shape=(2, L, n))
    capi.check(lib.he_rotate(h, L, da.ptr, ptrs, drot.ptr, elt, ws.ptr, None))
    assert (drot.numpy() == p.apply_galois(a, elt, host_evk)).all()
    # keys and digits
    out = DeviceArray(capi, shape=(2, L - 1, n))
    capi.check(lib.he_keyswitch_rescale(h, L, db.at(L * n), ptrs, da.ptr, out.ptr, 0, ws.ptr, None))
    assert (out.numpy() == p.rescale(want)).all()
    capi.check(lib.he_multiply_relin_rescale(h, L, da.ptr, db.ptr, ptrs, out.ptr, ws.ptr, None))
    assert (out.numpy() == p.rescale(p.relinearize(p.tensor(a, b), host_evk))).all()
