"""Calls at the ends of what the entry points take: more rows of sums than one launch or one call of the C-ABI holds."""
import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


def keys_for(cahel, parms, ctx):
    sk = cahel.secret_key(parms)
    sk.gen_secretkey(ctx)
    pk = cahel.public_key(ctx)
    sk.gen_publickey(ctx, pk)
    return sk, pk


@pytest.mark.parametrize("size,items", [(2, 16384), (4, 16384), (16, 4095), (16, 4096)])
def test_rows_of_sums_past_one_launch(oracle, capi, size, items):
    """he_sum_ciphertexts: a launch holds 65535 polynomials."""
    cahel, parms, ctx, p = make_pair(oracle, 9, [40, 40], 1)
    rng = np.random.default_rng(size)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    cts = [rand_limbs(p, rng, range(1), n_polys=size) for _ in range(3)]
    dev = [DeviceArray(capi, host=ct) for ct in cts]
    pick = rng.integers(0, 3, (items, 2))
    table = DeviceArray(capi, host=np.array([d.ptr for d in dev], dtype=np.uint64)[pick])
    out = DeviceArray(capi, shape=(items, size, 1, n))
    capi.check(lib.he_sum_ciphertexts(h, 1, size, items, 2, table.ptr, out.ptr, None))
    sums = np.array([[[p.add(cts[i][r], cts[j][r]) for r in range(size)] for j in range(3)] for i in range(3)])
    got = out.numpy()
    for i in range(3):
        for j in range(3):
            assert (got[(pick == [i, j]).all(axis=1)] == sums[i, j]).all(), (i, j)
    assert lib.he_sum_ciphertexts(h, 1, size, 16385, 2, table.ptr, out.ptr, None) == -1


@pytest.mark.parametrize("rows", [4096, 16384, 16385])
def test_any_number_of_rows(oracle, rows):
    """sum_ciphertexts and multiply_sum take as many rows as a loop of add and multiply does."""
    cahel, parms, ctx, p = make_pair(oracle, 9, [50, 40, 50], 1)
    sk, pk = keys_for(cahel, parms, ctx)
    enc = cahel.ckks_encoder(ctx)
    rng = np.random.default_rng(rows)
    a, b = (pk.encrypt_asymmetric(ctx, enc.encode(ctx, rng.uniform(-1, 1, p.n // 2), 2.0 ** 30)) for _ in range(2))
    ab, aa = p.tensor(a.to_numpy(), b.to_numpy()), p.tensor(a.to_numpy(), a.to_numpy())
    kinds = [[a, b], [a, a]]
    want_sum = [np.stack([p.add(x.to_numpy()[r], y.to_numpy()[r]) for r in range(2)]) for x, y in kinds]
    want_mul = [np.stack([p.add(aa[r], z[r]) for r in range(3)]) for z in (ab, aa)]
    which = [k % 2 for k in range(rows - 1)] + [1]
    sums = cahel.sum_ciphertexts(ctx, [kinds[k] for k in which])
    products = cahel.multiply_sum(ctx, [kinds[k] for k in which], [a, a])
    assert len(sums) == len(products) == rows
    for k in sorted({0, 1, 4094, 4095, rows - 3, rows - 2, rows - 1}):
        assert (sums[k].to_numpy() == want_sum[which[k]]).all(), k
        assert (products[k].to_numpy() == want_mul[which[k]]).all(), k
