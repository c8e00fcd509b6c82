"""Products whose last pass forms d0 and d1 from the factors, against the tensor product, key switch and rescale call by call, and against
themselves with a result that lies over a factor (which takes (d0, d1) from the workspace): the same words, on both sides of the line.  On
integers and on both arithmetics also against the oracle (FP64: test_gpu_fullsize.py)."""
import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu

CASES = [  # log_n, bits, size_p, L, items
    (13, [50] * 6 + [50] * 2, 2, 6, 11),              # FP64: 8.25 * 2^16 words a polynomial, and below the line
    (13, [50] * 6 + [50] * 2, 2, 6, 10),
    (14, [60] + [40] * 5 + [60] * 2, 2, 6, 6),        # both arithmetics
    (15, [60] + [40] * 3 + [60], 1, 4, 4),            # one special prime
    (14, [60] * 8 + [60] * 2, 2, 8, 8),               # integers: on the line
    (13, [60] * 8 + [60], 1, 7, 19),                  # one special prime, L < size_q
    (16, [50] * 12 + [50] * 4, 4, 10, 1),             # one product, a partial last digit
    (13, [60] + [40] * 5 + [60] * 2, 2, 6, 22),       # words that pass by the caches: from 16 * 2^16 on,
    (13, [50] * 6 + [50] * 2, 2, 6, 86),              # with the factors from 64 * 2^16
    (17, [50, 50], 1, 2, 2),                          # two limbs: one stays (the largest ring)
]


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


@pytest.mark.parametrize("square", [False, True])
@pytest.mark.parametrize("log_n,bits,size_p,L,items", CASES)
def test_products_equal_their_steps(oracle, capi, log_n, bits, size_p, L, items, square):
    bits = bits + [bits[-1]] * (L + size_p - len(bits))
    cahel, parms, ctx, p = make_pair(oracle, log_n, bits, size_p)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    rng = np.random.default_rng(log_n)
    keys = [DeviceArray(capi, host=rand_limbs(p, rng, range(p.size_qp), n_polys=2)) for _ in range(-(-p.size_q // size_p))]
    evk = capi.evk_array([k.ptr for k in keys])
    a = rand_limbs(p, rng, range(L), n_polys=2 * items)
    a[0, 0, :4] = [0, 1, p.moduli[0] - 1, p.moduli[0] - 2]
    b = a if square else rand_limbs(p, rng, range(L), n_polys=2 * items)
    da = DeviceArray(capi, host=a)
    db = da if square else DeviceArray(capi, host=b)
    ws = DeviceArray(capi, shape=(lib.he_multiply_relin_rescale_batch_workspace_words(h, L, items),))
    out = DeviceArray(capi, shape=(items, 2, L - 1, n))
    capi.check(lib.he_multiply_relin_rescale_batch(h, L, items, da.ptr, db.ptr, evk, out.ptr, ws.ptr, None))
    got = out.numpy()
    assert (da.numpy() == a).all()
    over = DeviceArray(capi, host=a)
    capi.check(lib.he_multiply_relin_rescale_batch(h, L, items, over.ptr, over.ptr if square else db.ptr, evk, over.ptr, ws.ptr, None))
    assert (over.numpy().reshape(-1)[:got.size] == got.reshape(-1)).all()
    one = DeviceArray(capi, shape=(2, L - 1, n))
    d = DeviceArray(capi, shape=(3, L, n))
    for k in sorted({0, items // 2, items - 1}):
        at = 2 * k * L * n
        capi.check(lib.he_tensor(h, da.at(at), db.at(at), d.ptr, L, None))
        capi.check(lib.he_keyswitch_rescale(h, L, d.at(2 * L * n), evk, d.ptr, one.ptr, 0, ws.ptr, None))
        assert (got[k] == one.numpy()).all(), k


@pytest.mark.parametrize("log_n,bits,size_p,L,items", [(13, [60] * 8 + [60] * 2, 2, 8, 16),             # integers: on the line, 2^20 words
                                                        (15, [60] * 6 + [60], 1, 6, 6),                  # one special prime
                                                        (14, [60] + [40] * 5 + [60] * 2, 2, 6, 6),       # both arithmetics
                                                        (16, [50] * 4 + [50] * 2, 2, 4, 4),              # FP64: on the line
                                                        (16, [60] + [40] * 11 + [60] * 4, 4, 12, 2),     # both: twiddles worked out, the fewest
                                                        (16, [60] + [40] * 11 + [60] * 4, 4, 11, 2)])    # ... and read
def test_products_equal_the_oracle(oracle, capi, log_n, bits, size_p, L, items):
    cahel, parms, ctx, p = make_pair(oracle, log_n, bits, size_p)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    assert items * L << log_n >= (16 if bits[1] > 50 else 8) << 16
    rng = np.random.default_rng(log_n)
    host_evk = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(p.size_q // size_p)]
    dev_evk = [DeviceArray(capi, host=k) for k in host_evk]
    evk = capi.evk_array([k.ptr for k in dev_evk])
    a, b = (np.stack([rand_limbs(p, rng, range(L), n_polys=2) for _ in range(items)]) for _ in range(2))
    a[0, 0, 0, :4] = b[-1, 1, 0, :4] = [0, 1, p.moduli[0] - 1, p.moduli[0] - 2]
    da, db = DeviceArray(capi, host=a), DeviceArray(capi, host=b)
    ws = DeviceArray(capi, shape=(lib.he_multiply_relin_rescale_batch_workspace_words(h, L, items),))
    out = DeviceArray(capi, shape=(items, 2, L - 1, n))
    for x, y, dx, dy in ((a, b, da, db), (b, b, db, db)):
        capi.check(lib.he_multiply_relin_rescale_batch(h, L, items, dx.ptr, dy.ptr, evk, out.ptr, ws.ptr, None))
        got = out.numpy()
        for k in sorted({0, items // 2, items - 1}):
            assert (got[k] == p.rescale(p.relinearize(p.tensor(x[k], y[k]), host_evk))).all(), k
