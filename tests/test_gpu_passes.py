"""Edges of the transform passes and of what is fused with them, against the oracle: batches on both sides of the sizes at
which a launch changes its tile or walks several limbs per wave, the encoding that forms no maximum, encryption and decryption
from byte samples, and the decoding that is composed where the inverse transform ends; on all three back ends."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import DeviceArray, make_pair, rand_limbs

pytestmark = pytest.mark.gpu

CHAINS = {"fp": [50, 49, 50, 48, 50, 50], "int": [60, 58, 60, 60, 55, 60], "mixed": [60, 40, 40, 50, 60, 60]}


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,limbs,polys", [(15, 5, 30), (15, 5, 41), (16, 4, 7), (16, 4, 8), (16, 1, 1)])
def test_batched_transforms(oracle, capi, chain, logn, limbs, polys):
    cahel, parms, ctx, p = make_pair(oracle, logn, CHAINS[chain], 1)
    lib, h = capi.lib(), ctx.he_handle()
    x = rand_limbs(p, np.random.default_rng(polys), range(limbs), n_polys=polys)
    x[0, 0, :4] = [0, 1, p.moduli[0] - 1, p.moduli[0] - 2]
    d = DeviceArray(capi, host=x)
    capi.check(lib.he_ntt_forward(h, d.ptr, polys, limbs, limbs, 0, limbs, 0, None))
    got = d.numpy()
    for k in sorted({0, 1, polys // 2, polys - 1} & set(range(polys))):
        assert (got[k] == p.ntt_fwd(x[k].copy())).all(), k
    capi.check(lib.he_ntt_inverse(h, d.ptr, polys, limbs, limbs, 0, limbs, 0, None))
    assert (d.numpy() == x).all()


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,limbs,polys", [(10, 1, 1), (10, 5, 3), (12, 1, 1), (12, 3, 53), (12, 5, 32), (12, 5, 51), (12, 5, 52), (13, 5, 25),
                                              (13, 4, 32)])
@pytest.mark.parametrize("one_pass", ["default", "forced"])
def test_whole_limb_transforms(oracle, capi, monkeypatch, chain, logn, limbs, polys, one_pass):
    """A limb of 2^10, 2^12 or 2^13 words in one workgroup, on both sides of the numbers of limbs at which it begins to run at 2^12
    (integers, 159 and 160) and 2^13 (125 and 128) and at which the kernel changes at 2^12 (255 and 260)."""
    monkeypatch.setenv("CAHEL_HIP_FORCE_ONE_PASS", "1" if one_pass == "forced" else "0")
    cahel, parms, ctx, p = make_pair(oracle, logn, CHAINS[chain], 1)
    lib, h = capi.lib(), ctx.he_handle()
    x = rand_limbs(p, np.random.default_rng(polys), range(limbs), n_polys=polys)
    x[0, 0, :4] = [0, 1, p.moduli[0] - 1, p.moduli[0] - 2]
    x[polys - 1, limbs - 1, :] = p.moduli[limbs - 1] - 1
    d = DeviceArray(capi, host=x)
    capi.check(lib.he_ntt_forward(h, d.ptr, polys, limbs, limbs, 0, limbs, 0, None))
    got = d.numpy()
    for k in sorted({0, polys // 2, polys - 1}):
        assert (got[k] == p.ntt_fwd(x[k].copy())).all(), k
    capi.check(lib.he_ntt_inverse(h, d.ptr, polys, limbs, limbs, 0, limbs, 0, None))
    assert (d.numpy() == x).all()


@pytest.mark.parametrize("bits", [60, 50, 49, 30])
@pytest.mark.parametrize("logn,limbs", [(9, 2), (11, 2), (13, 2), (16, 2), (16, 18), (17, 2), (17, 9)])
def test_passes_of_the_largest_words(oracle, capi, monkeypatch, logn, limbs, bits):
    """Lazy ranges of both back ends, primes at the ends of FP64's; words of q - 1 throughout, and random ones.  FP64 passes over 36 * 2^16
    words and more work out the twiddles of their last two stages from two entries of the table: every block of the limb."""
    monkeypatch.setenv("CAHEL_HIP_NO_ONE_PASS", "1")
    cahel, parms, ctx, p = make_pair(oracle, logn, [bits] * (limbs + 1), 1)
    lib, h = capi.lib(), ctx.he_handle()
    x = rand_limbs(p, np.random.default_rng(logn), range(limbs), n_polys=2)
    for i in range(limbs):
        x[1, i, :] = p.moduli[i] - 1
    d = DeviceArray(capi, host=x)
    capi.check(lib.he_ntt_forward(h, d.ptr, 2, limbs, limbs, 0, limbs, 0, None))
    got = d.numpy()
    assert all((got[k] == p.ntt_fwd(x[k].copy())).all() for k in range(2))
    capi.check(lib.he_memcpy_h2d(d.ptr, x.ctypes.data, x.nbytes, None))
    capi.check(lib.he_ntt_inverse(h, d.ptr, 2, limbs, limbs, 0, limbs, 0, None))
    got = d.numpy()
    assert all((got[k] == p.ntt_inv(x[k].copy())).all() for k in range(2))


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,size_p,L", [(12, 1, 5), (13, 2, 3), (14, 1, 1), (15, 2, 4), (16, 1, 2)])
def test_encrypt_and_decrypt(oracle, capi, chain, logn, size_p, L):
    """he_encrypt of a plaintext elsewhere, he_encrypt_batch of three in place, he_decrypt_flood of 2 and 3 polynomials."""
    cahel, parms, ctx, p = make_pair(oracle, logn, CHAINS[chain], size_p)
    lib, h = capi.lib(), ctx.he_handle()
    rng = np.random.default_rng(logn)
    n, Q, K, items, first = p.n, p.size_q, p.size_p, 3, 11
    key = oracle.chacha_key(3)
    kp = key.ctypes.data_as(C.POINTER(C.c_uint32))
    pk = rand_limbs(p, rng, range(p.size_qp), n_polys=2)
    plain = rand_limbs(p, rng, range(L), n_polys=items)
    dpk, dplain = DeviceArray(capi, host=pk), DeviceArray(capi, host=plain)
    cts = np.zeros((items, 2, L, n), dtype=np.uint64)
    cts[:, 0] = plain
    dcts, dct = DeviceArray(capi, host=cts), DeviceArray(capi, shape=(2, L, n))
    ws = DeviceArray(capi, shape=(lib.he_encrypt_batch_workspace_words(h, L, items),))
    capi.check(lib.he_encrypt_batch(h, L, items, dpk.ptr, kp, first, dcts.ptr, ws.ptr, None))
    capi.check(lib.he_encrypt(h, L, dplain.at(L * n), dpk.ptr, kp, first + 3, dct.ptr, ws.ptr, None))
    got = dcts.numpy()
    assert (dct.numpy() == got[1]).all()
    # the oracle's division works on L + K limbs: those of Q that are in use, then the special ones
    tidx = list(range(L)) + list(range(Q, Q + K))
    for k in range(items):
        u = p.ntt_fwd(p.sample_ternary(key, first + 3 * k, p.size_qp))
        for i in range(2):
            e = p.ntt_fwd(p.sample_error(key, first + 3 * k + 1 + i, p.size_qp))
            want = p.moddown(np.ascontiguousarray(p.mul_add(u, pk[i], e)[tidx]))
            assert (got[k, i] == (p.add(want, plain[k]) if i == 0 else want)).all(), (k, i)
    cdt = oracle.gauss_cdt()
    dcdt, noise = DeviceArray(capi, host=cdt), DeviceArray(capi, shape=(n // 8,))
    sk = rand_limbs(p, rng, range(L), n_polys=2)
    ct = rand_limbs(p, rng, range(L), n_polys=3)
    dsk, dct3, out = DeviceArray(capi, host=sk), DeviceArray(capi, host=ct), DeviceArray(capi, shape=(L, n))
    e = p.ntt_fwd(p.sample_gauss(key, 5, L, cdt))
    for size in (2, 3):
        capi.check(lib.he_decrypt_flood(h, dct3.ptr, size, L, dsk.ptr, L * n, kp, 5, dcdt.ptr, len(cdt), out.ptr, noise.ptr, None))
        want = p.mul_add(ct[1], sk[0], ct[0])
        want = p.mul_add(ct[2], sk[1], want) if size == 3 else want
        assert (out.numpy() == p.add(want, e)).all(), size
    assert lib.he_decrypt_flood(h, dct3.ptr, 4, L, dsk.ptr, L * n, kp, 5, dcdt.ptr, len(cdt), out.ptr, noise.ptr, None) != 0
    assert lib.he_decrypt_flood(h, dct3.ptr, 2, L, dsk.ptr, L * n, kp, 5, dcdt.ptr, 128, out.ptr, noise.ptr, None) != 0


@pytest.mark.parametrize("slots", [128, 256, 512, 1024, 2048])
def test_slot_transform_at_the_edges_of_its_rows(oracle, capi, slots):
    """Encoding and decoding where the special FFT changes its shape: inside LDS, one block of 256, two of them, one block of
    1024, two of them.  Coefficients within one unit of the oracle's (the rounding of a sum that falls on the middle), values
    within 2^-20: 12 stages in double precision and a rounding to 2^-41 per coefficient stay far below."""
    cahel, parms, ctx, p = make_pair(oracle, 12, CHAINS["mixed"], 1)
    lib, h = capi.lib(), ctx.he_handle()
    rng = np.random.default_rng(slots)
    limbs, n, count, scale = 2, p.n, slots - 3, 2.0 ** 40
    z = rng.uniform(-1, 1, count) + 1j * rng.uniform(-1, 1, count)
    o_enc = oracle.Encoder(p)
    re, im = DeviceArray(capi, host=np.ascontiguousarray(z.real)), DeviceArray(capi, host=np.ascontiguousarray(z.imag))
    ws, out = DeviceArray(capi, shape=(lib.he_ckks_workspace_words(h, limbs),)), DeviceArray(capi, shape=(limbs, n))
    capi.check(lib.he_ckks_encode(h, re.ptr, im.ptr, count, slots, scale, limbs, out.ptr, ws.ptr, None))
    got = out.numpy()
    got_coeff, want_coeff = p.ntt_inv(got.copy()), p.ntt_inv(o_enc.encode(z, scale, limbs, slots))
    for i in range(limbs):
        q = p.moduli[i]
        d = (got_coeff[i].astype(np.int64) - want_coeff[i].astype(np.int64)) % q
        assert np.minimum(d, q - d).max() <= 1, i
    dec = DeviceArray(capi, shape=(slots, 2), dtype=np.float64)
    capi.check(lib.he_ckks_decode(h, out.ptr, limbs, slots, scale, dec.ptr, ws.ptr, None))
    values = dec.numpy() @ np.array([1, 1j])
    assert np.abs(values - o_enc.decode(got, scale, slots)).max() < 2.0 ** -20
    assert np.abs(values[:count] - z).max() < 2.0 ** -20 and np.abs(values[count:]).max() < 2.0 ** -20


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,slots,limbs", [(12, 2, 1), (12, 2048, 5), (13, 128, 2), (13, 4096, 3), (14, 512, 4), (15, 16384, 2),
                                              (16, 32768, 4), (17, 65536, 2)])
def test_bounded_encoding_and_real_decoding(oracle, capi, chain, logn, slots, limbs):
    """he_ckks_encode_bounded gives he_ckks_encode_batch's plaintexts, up to the largest coefficients it is for;
    he_ckks_decode_real and he_decrypt_decode_real_batch give he_ckks_decode's real parts."""
    cahel, parms, ctx, p = make_pair(oracle, logn, CHAINS[chain], 1)
    lib, h = capi.lib(), ctx.he_handle()
    rng = np.random.default_rng(slots)
    items, n, count, scale = 2, p.n, slots - slots // 3, 2.0 ** 40
    z = rng.uniform(-1, 1, (2, items, count)) * np.array([2.0 ** 20, 1.0])[None, :, None]
    z[:, 0] *= slots / count / 2.0                 # item 0: sums of magnitudes below 2^20 slots, coefficients up to 2^60
    re, im = DeviceArray(capi, host=z[0]), DeviceArray(capi, host=z[1])
    ws = DeviceArray(capi, shape=(lib.he_ckks_encode_batch_workspace_words(h, items),))
    want, got = (DeviceArray(capi, host=np.zeros((items, limbs, n), dtype=np.uint64)) for _ in range(2))
    capi.check(lib.he_ckks_encode_batch(h, re.ptr, im.ptr, count, slots, scale, limbs, items, count, want.ptr, limbs, ws.ptr, None))
    capi.check(lib.he_ckks_encode_bounded(h, re.ptr, im.ptr, count, slots, scale, limbs, items, count, got.ptr, limbs, ws.ptr, None))
    plain = want.numpy()
    assert (got.numpy() == plain).all()
    # ciphertexts (plain, 0): whatever the key, they decrypt to the plaintext
    cts = np.zeros((items, 2, limbs, n), dtype=np.uint64)
    cts[:, 0] = plain
    dcts, sk = DeviceArray(capi, host=cts), DeviceArray(capi, host=np.ones((limbs, n), dtype=np.uint64))
    table = DeviceArray(capi, host=np.array([dcts.at(k * 2 * limbs * n) for k in range(items)], dtype=np.uint64))
    take = max(1, slots - 1)
    dws = DeviceArray(capi, shape=(lib.he_ckks_workspace_words(h, limbs),))
    rws = DeviceArray(capi, shape=(lib.he_decrypt_decode_real_workspace_words(h, limbs, slots, items),))
    full, real = DeviceArray(capi, shape=(slots, 2), dtype=np.float64), DeviceArray(capi, shape=(items, take), dtype=np.float64)
    capi.check(lib.he_decrypt_decode_real_batch(h, table.ptr, items, limbs, sk.ptr, None, 0, None, 0, slots, scale, take, real.ptr,
                                                rws.ptr, None))
    batch = real.numpy()
    for k in range(items):
        capi.check(lib.he_ckks_decode(h, want.at(k * limbs * n), limbs, slots, scale, full.ptr, dws.ptr, None))
        capi.check(lib.he_ckks_decode_real(h, want.at(k * limbs * n), limbs, slots, scale, real.ptr, take, rws.ptr, None))
        values = full.numpy()[:take, 0]
        assert (real.numpy()[0] == values).all() and (batch[k] == values).all(), k
        if limbs > 1 or k == 1:
            assert np.abs(values[:count] - z[0, k][:take]).max() < 2.0 ** -18, k


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,size_p,L,n_steps", [(9, 1, 4, 1), (9, 2, 3, 40), (12, 2, 4, 1), (12, 2, 3, 2), (13, 1, 5, 1), (14, 1, 4, 16),
                                                   (16, 2, 4, 3)])
def test_hoisting_of_one_ciphertext(oracle, capi, chain, logn, size_p, L, n_steps):
    """he_hoisted_rotations with fewer, as many and more terms than the waves that share a block (3, 4, 5: one is left without),
    in one launch and in several that add up, with and without the input added."""
    cahel, parms, ctx, p = make_pair(oracle, logn, CHAINS[chain], size_p)
    rng = np.random.default_rng(n_steps)
    lib, h = capi.lib(), ctx.he_handle()
    beta = -(-L // size_p)
    host = [[rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(beta)] for _ in range(2)]
    dev = [[DeviceArray(capi, host=d) for d in key] for key in host]
    # elements of every residue modulo 4 and 8: neighbouring words keep their order or are turned round
    elts = [(pow(5, 3 * k + 1, 2 * p.n) * (2 * p.n - 1 if k % 2 else 1)) % (2 * p.n) for k in range(n_steps)]
    flat = capi.evk_array([dev[i % 2][d].ptr for i in range(n_steps) for d in range(beta)])
    d_elts = (C.c_uint32 * n_steps)(*elts)
    ws = DeviceArray(capi, shape=(lib.he_keyswitch_batch_workspace_words(h, L, 1),))
    ct = rand_limbs(p, rng, range(L), n_polys=2)
    want = p.hoisting(ct, elts, [host[i % 2] for i in range(n_steps)])
    din, dout = DeviceArray(capi, host=ct), DeviceArray(capi, shape=(2, L, p.n))
    capi.check(lib.he_hoisted_rotations(h, L, din.ptr, flat, d_elts, n_steps, dout.ptr, ws.ptr, None))
    assert (dout.numpy() == want).all()
    capi.check(lib.he_hoisted_rotations_batch(h, L, 1, din.ptr, flat, d_elts, n_steps, 1, dout.ptr, ws.ptr, None))
    assert (dout.numpy() == np.stack([p.add(want[i], ct[i]) for i in range(2)])).all()
    assert (din.numpy() == ct).all()


@pytest.mark.parametrize("logn,bits,size_p,levels", [
    (12, [60, 40, 60, 40, 60, 40, 60, 60], 2, (6, 3)), (13, [60, 58, 60, 60, 55, 60, 60, 60, 60], 3, (6, 5)),
    (14, [60, 45, 45, 45, 60, 60, 60, 60], 4, (4, 2)), (15, [60, 40, 40, 40, 40, 60, 60, 60, 60, 60], 5, (5, 4)),
    (16, [60, 40, 60, 50, 60, 60], 2, (4, 3)), (16, [60] * 4 + [50] * 4 + [60] * 8, 8, (8,))])
def test_conversion_fused_on_integers(oracle, capi, logn, bits, size_p, levels):
    """ModUp, ModDown and the merged ModDown + rescale of levels with primes from 2^50 on, of up to 4 and up to 8 input limbs a
    digit, with residues that make the largest sums, and of a batch."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, size_p)
    rng = np.random.default_rng(logn)
    lib, h = capi.lib(), ctx.he_handle()
    K, n, items = p.size_p, p.n, 3
    host = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(p.size_q // K)]
    dev = [DeviceArray(capi, host=k) for k in host]
    ptrs = capi.evk_array([d.ptr for d in dev])
    for L in levels:
        beta, tables = -(-L // K), [p.table_index(L, t) for t in range(L + K)]
        dy, ws = DeviceArray(capi, shape=(beta, L + K, n)), DeviceArray(capi, shape=(2 * L, n))
        coeff = np.stack([np.full(n, p.moduli[t] - 1, dtype=np.uint64) for t in range(L)])
        for c in (rand_limbs(p, rng, range(L)), p.ntt_fwd(coeff, list(range(L)))):
            dc = DeviceArray(capi, host=c)
            capi.check(lib.he_modup(h, L, dc.ptr, dy.ptr, ws.ptr, None))
            assert (dy.numpy() == p.modup(c)).all(), L
        cx = np.stack([rand_limbs(p, rng, tables) for _ in range(2)])
        dcx, dout, wsd = DeviceArray(capi, host=cx), DeviceArray(capi, shape=(2, L, n)), DeviceArray(capi, shape=(2, L, n))
        capi.check(lib.he_moddown(h, L, dcx.ptr, dout.ptr, 2, 0, wsd.ptr, None))
        assert (dout.numpy() == np.stack([p.moddown(x) for x in cx])).all(), L
        c = rand_limbs(p, rng, range(L), n_polys=items)
        ct = np.stack([rand_limbs(p, rng, range(L), n_polys=2) for _ in range(items)])
        dc, dct, out = DeviceArray(capi, host=c), DeviceArray(capi, host=ct), DeviceArray(capi, shape=(items, 2, L - 1, n))
        bws = DeviceArray(capi, shape=(lib.he_keyswitch_batch_workspace_words(h, L, items),))
        capi.check(lib.he_keyswitch_rescale_batch(h, L, items, dc.ptr, L, ptrs, dct.ptr, out.ptr, 0, bws.ptr, None))
        got = out.numpy()
        for k in range(items):
            ks = p.key_switch(c[k], host)
            assert (got[k] == p.rescale(np.stack([p.add(ct[k][b], ks[b]) for b in range(2)]))).all(), (L, k)


@pytest.mark.parametrize("chain", sorted(CHAINS) + ["largest"])
@pytest.mark.parametrize("logn,L,items,count", [(9, 1, 1, 1), (10, 5, 3, 2), (13, 2, 2, 16), (12, 3, 1, 17), (16, 2, 2, 33)])
def test_sums_of_ciphertexts_and_products(oracle, capi, chain, logn, L, items, count):
    """he_sum_ciphertexts and he_multiply_sum around the 16 terms after which the products' sums are reduced, some of the words
    the largest residues, some operands shared between the sums."""
    cahel, parms, ctx, p = make_pair(oracle, logn, CHAINS.get(chain, [60] * 6), 1)
    rng = np.random.default_rng(count)
    lib, h = capi.lib(), ctx.he_handle()
    n, kinds = p.n, min(3, count + 1)
    top = np.array(p.moduli[:L], dtype=np.uint64)[:, None] - np.uint64(1)
    cts = [rand_limbs(p, rng, range(L), n_polys=2) for _ in range(kinds)]
    for ct in cts:
        ct[:, :, :n // 2] = top
    dev = [DeviceArray(capi, host=ct) for ct in cts]
    pick = rng.integers(0, kinds, (items, count, 2))
    table = DeviceArray(capi, host=np.array([[[dev[i].at(0) for i in pair] for pair in row] for row in pick], dtype=np.uint64))
    first = DeviceArray(capi, host=np.array([[dev[pair[0]].at(0) for pair in row] for row in pick], dtype=np.uint64))
    out, products = DeviceArray(capi, shape=(items, 2, L, n)), DeviceArray(capi, shape=(items, 3, L, n))
    capi.check(lib.he_sum_ciphertexts(h, L, 2, items, count, first.ptr, out.ptr, None))
    capi.check(lib.he_multiply_sum(h, L, items, count, table.ptr, products.ptr, None))
    got, got3 = out.numpy(), products.numpy()
    tensors = {(i, j): p.tensor(cts[i], cts[j]) for i, j in {tuple(x) for row in pick for x in row}}
    for k in range(items):
        want, want3 = cts[pick[k, 0, 0]], tensors[tuple(pick[k, 0])]
        for i, j in pick[k, 1:]:
            want = np.stack([p.add(want[r], cts[i][r]) for r in range(2)])
            want3 = np.stack([p.add(want3[r], tensors[(i, j)][r]) for r in range(3)])
        assert (got[k] == want).all() and (got3[k] == want3).all(), k
    assert lib.he_sum_ciphertexts(h, L, 2, items, 0, first.ptr, out.ptr, None) == -1
    assert lib.he_multiply_sum(h, 7, items, count, table.ptr, products.ptr, None) == -1


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("local", [False, True])
@pytest.mark.parametrize("logn,size_p,L,n_steps,items", [(9, 1, 1, 1, 2), (10, 1, 3, 3, 3), (12, 2, 4, 4, 4), (11, 1, 4, 16, 5), (13, 1, 1, 17, 6),
                                                         (16, 1, 2, 15, 5)])
def test_hoisting_of_batches(oracle, capi, chain, local, logn, size_p, L, n_steps, items):
    """he_hoisted_rotations_batch with odd and even counts of terms around the 8 after which the integer sums are relieved (up to
    64 of them), with groups of two and of four ciphertexts and a rest, with keys that make the largest partial products and
    differences (halves all ones or zero), steps inside aligned blocks and across them."""
    cahel, parms, ctx, p = make_pair(oracle, logn, CHAINS[chain], size_p)
    rng = np.random.default_rng(n_steps)
    lib, h = capi.lib(), ctx.he_handle()
    beta = -(-L // size_p)
    host = [[rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(beta)] for _ in range(2)]
    for key in host[0]:
        for t in range(p.size_qp):
            q, low = p.moduli[t], (1 << 30) - 1
            key[:, t, :4] = [q - 1, low, (q - 1) & ~low, 0]
            key[0, t, 4:p.n // 2] = min(low, q - 1)
            key[1, t, 4:p.n // 2] = (q - 1) & ~low
    dev = [[DeviceArray(capi, host=d) for d in key] for key in host]
    unit = max(1, p.n // 512) if local else 1
    elts = [pow(5, unit * (k + 1), 2 * p.n) for k in range(n_steps)]
    flat = capi.evk_array([dev[i % 2][d].ptr for i in range(n_steps) for d in range(beta)])
    d_elts = (C.c_uint32 * n_steps)(*elts)
    wsb = DeviceArray(capi, shape=(lib.he_keyswitch_batch_workspace_words(h, L, items),))
    cts = np.stack([rand_limbs(p, rng, range(L), n_polys=2) for _ in range(items)])
    din, dout = DeviceArray(capi, host=cts), DeviceArray(capi, shape=(items, 2, L, p.n))
    want = [p.hoisting(ct, elts, [host[i % 2] for i in range(n_steps)]) for ct in cts]
    for add_input in (0, 1):
        capi.check(lib.he_hoisted_rotations_batch(h, L, items, din.ptr, flat, d_elts, n_steps, add_input, dout.ptr, wsb.ptr, None))
        got = dout.numpy()
        for k in range(items):
            w = np.stack([p.add(want[k][b], cts[k][b]) for b in range(2)]) if add_input else want[k]
            assert (got[k] == w).all(), (add_input, k)
    assert (din.numpy() == cts).all()


@pytest.mark.parametrize("logn,bits,size_p,L", [(16, [60, 40, 40, 60], 1, 2), (16, [60, 40, 40, 60], 1, 3), (15, [40, 60, 50, 45, 30, 59, 60, 50], 2, 5),
                                                (15, [60, 40, 50, 45, 30, 59, 60, 60], 2, 4), (14, [60, 40, 50, 45, 30, 59, 60, 60], 2, 6),
                                                (12, [60, 40, 60], 1, 2), (13, [60, 40, 50, 45, 60], 1, 3),
                                                (13, [60] + [40] * 23 + [60] * 8, 8, 24), (14, [60] + [40] * 15 + [60] * 4, 4, 15)])
def test_key_switch_of_a_mixed_chain(oracle, capi, logn, bits, size_p, L):
    """Rotation and key switch + rescale where the inner product takes its limbs in an order of their own (more than one workgroup for
    every CU) and where it does not, with even and odd numbers of primes (behind an odd one the constants of P lie a word further), with an epilogue's workgroups dealt to all
    XCDs (768 and more) and not."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, size_p)
    rng = np.random.default_rng(logn + L)
    lib, h = capi.lib(), ctx.he_handle()
    host = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(p.size_q // p.size_p)]
    dev = [DeviceArray(capi, host=k) for k in host]
    keys = capi.evk_array([d.ptr for d in dev])
    ws = DeviceArray(capi, shape=(lib.he_keyswitch_workspace_words(h, L),))
    ct, c = rand_limbs(p, rng, range(L), n_polys=2), rand_limbs(p, rng, range(L))
    dct, dc = DeviceArray(capi, host=ct), DeviceArray(capi, host=c)
    out, elt = DeviceArray(capi, shape=(2, L, p.n)), 25
    capi.check(lib.he_rotate(h, L, dct.ptr, keys, out.ptr, elt, ws.ptr, None))
    ks = p.key_switch(p.galois_ntt(ct[1], elt), host)
    assert (out.numpy() == np.stack([p.add(p.galois_ntt(ct[0], elt), ks[0]), ks[1]])).all()
    low = DeviceArray(capi, shape=(2, L - 1, p.n))
    capi.check(lib.he_keyswitch_rescale(h, L, dc.ptr, keys, dct.ptr, low.ptr, 0, ws.ptr, None))
    ks = p.key_switch(c, host)
    assert (low.numpy() == p.rescale(np.stack([p.add(ct[b], ks[b]) for b in range(2)]))).all()


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("size_p,L", [(1, 2), (1, 3), (1, 4), (1, 5), (2, 2), (2, 3), (2, 4)])
def test_key_switches_of_few_and_of_many_digits(oracle, capi, chain, size_p, L):
    """The inner product takes its keys' addresses in one form up to three digits of one ciphertext and in another beyond; the converted
    limbs of a digit (the last one may have fewer) are worked out.  A map of one run may have anything as its second run."""
    cahel, parms, ctx, p = make_pair(oracle, 13, CHAINS[chain], size_p)
    rng = np.random.default_rng(16 * size_p + L)
    lib, h = capi.lib(), ctx.he_handle()
    host = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(-(-p.size_q // p.size_p))]
    dev = [DeviceArray(capi, host=k) for k in host]
    keys = capi.evk_array([d.ptr for d in dev])
    for items in (1, 2):
        cs = np.stack([rand_limbs(p, rng, range(L)) for _ in range(items)])
        cts = np.stack([rand_limbs(p, rng, range(L), n_polys=2) for _ in range(items)])
        dc, dct = DeviceArray(capi, host=cs), DeviceArray(capi, host=cts)
        low = DeviceArray(capi, shape=(items, 2, L - 1, p.n))
        ws = DeviceArray(capi, shape=(lib.he_keyswitch_batch_workspace_words(h, L, items),))
        capi.check(lib.he_keyswitch_rescale_batch(h, L, items, dc.ptr, L, keys, dct.ptr, low.ptr, 0, ws.ptr, None))
        got = low.numpy()
        for k in range(items):
            ks = p.key_switch(cs[k], host)
            assert (got[k] == p.rescale(np.stack([p.add(cts[k][b], ks[b]) for b in range(2)]))).all(), (items, k)
    x = rand_limbs(p, rng, range(L))
    d = DeviceArray(capi, host=x)
    capi.check(lib.he_ntt_forward(h, d.ptr, 1, L, L, 0, L, 0xfffffff7, None))
    assert (d.numpy() == p.ntt_fwd(x.copy())).all()
    capi.check(lib.he_ntt_inverse(h, d.ptr, 1, L, L, 0, L, 0xfffffff7, None))
    assert (d.numpy() == x).all()


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,limbs", [(11, 2), (12, 1), (12, 63), (13, 32), (13, 33), (14, 16), (14, 17), (15, 3), (16, 4), (16, 5)])
def test_decryption_where_the_noise_has_a_launch_of_its_own_and_where_not(oracle, capi, chain, logn, limbs):
    """Up to 2^18 coefficients the rows pass samples what it transforms."""
    bits = (CHAINS[chain] * 11)[:limbs + 1]
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, 1)
    lib, h, rng = capi.lib(), ctx.he_handle(), np.random.default_rng(logn + limbs)
    key, cdt = oracle.chacha_key(3), oracle.gauss_cdt()
    kp = key.ctypes.data_as(C.POINTER(C.c_uint32))
    ct, s = rand_limbs(p, rng, range(limbs), n_polys=2), rand_limbs(p, rng, range(limbs))
    dct, dsk, dcdt = DeviceArray(capi, host=ct), DeviceArray(capi, host=s), DeviceArray(capi, host=cdt)
    out, noise = DeviceArray(capi, shape=(limbs, p.n)), DeviceArray(capi, shape=(p.n // 8,))
    capi.check(lib.he_decrypt_flood(h, dct.ptr, 2, limbs, dsk.ptr, limbs * p.n, kp, 2 ** 40 + 5, dcdt.ptr, len(cdt), out.ptr, noise.ptr, None))
    assert (out.numpy() == p.add(p.mul_add(ct[1], s, ct[0]), p.ntt_fwd(p.sample_gauss(key, 2 ** 40 + 5, limbs, cdt)))).all()


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,L,items", [(11, 3, 1), (12, 2, 1), (13, 5, 3), (14, 4, 8), (14, 4, 10), (15, 8, 1), (15, 9, 1), (16, 4, 1), (16, 5, 1)])
def test_key_switch_and_rescale_of_few_limbs(oracle, capi, chain, logn, L, items):
    """One special prime: up to 7 * 2^16 output words the forward pass starts with the inverse passes of the dropped and the special limb."""
    bits = (CHAINS[chain] * 2)[:L + 1]
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, 1)
    rng = np.random.default_rng(logn + L)
    lib, h = capi.lib(), ctx.he_handle()
    host = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(2)]
    dev = [DeviceArray(capi, host=k) for k in host]
    keys = capi.evk_array([dev[d % 2].ptr for d in range(p.size_q)])
    cs, cts = rand_limbs(p, rng, range(L), n_polys=items), rand_limbs(p, rng, range(L), n_polys=2 * items).reshape(items, 2, L, p.n)
    cs[0, :, 0], cts[0, 0, :, 0] = [q - 1 for q in p.moduli[:L]], [q - 1 for q in p.moduli[:L]]
    dc, dct, low = DeviceArray(capi, host=cs), DeviceArray(capi, host=cts), DeviceArray(capi, shape=(items, 2, L - 1, p.n))
    ws = DeviceArray(capi, shape=(lib.he_keyswitch_batch_workspace_words(h, L, items),))
    capi.check(lib.he_keyswitch_rescale_batch(h, L, items, dc.ptr, L, keys, dct.ptr, low.ptr, 0, ws.ptr, None))
    got = low.numpy()
    for k in sorted({0, items - 1}):
        ks = p.key_switch(cs[k], [host[d % 2] for d in range(p.size_q)])
        assert (got[k] == p.rescale(np.stack([p.add(cts[k][b], ks[b]) for b in range(2)]))).all(), k


@pytest.mark.parametrize("size_p,L,items", [(4, 4, 8), (5, 10, 3), (5, 10, 4), (6, 12, 4), (8, 8, 8)])
def test_conversions_on_both_sides_of_the_matrix_kernel(oracle, capi, size_p, L, items):
    """Key switch + rescale at n = 2^16, primes below 2^50: from five special primes and 256 tiles on the conversions run on the matrix
    cores."""
    cahel, parms, ctx, p = make_pair(oracle, 16, [50] * (L + size_p), size_p)
    rng = np.random.default_rng(size_p + items)
    lib, h = capi.lib(), ctx.he_handle()
    host = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(2)]
    dev = [DeviceArray(capi, host=k) for k in host]
    beta = L // size_p
    keys = capi.evk_array([dev[d % 2].ptr for d in range(beta)])
    one, ct1 = rand_limbs(p, rng, range(L), n_polys=2), rand_limbs(p, rng, range(L), n_polys=2)
    one[0, :, :2] = np.array([[q - 1, 0] for q in p.moduli[:L]], dtype=np.uint64)
    cs, cts = np.stack([one[k % 2] for k in range(items)]), np.stack([ct1] * items)
    dc, dct, low = DeviceArray(capi, host=cs), DeviceArray(capi, host=cts), DeviceArray(capi, shape=(items, 2, L - 1, p.n))
    ws = DeviceArray(capi, shape=(lib.he_keyswitch_batch_workspace_words(h, L, items),))
    capi.check(lib.he_keyswitch_rescale_batch(h, L, items, dc.ptr, L, keys, dct.ptr, low.ptr, 0, ws.ptr, None))
    got = low.numpy()
    want = []
    for k in range(2):
        ks = p.key_switch(one[k], [host[d % 2] for d in range(beta)])
        want.append(p.rescale(np.stack([p.add(ct1[b], ks[b]) for b in range(2)])))
    for k in range(items):
        assert (got[k] == want[k % 2]).all(), k


@pytest.mark.parametrize("logn,L,size_p,items", [(14, 3, 1, 1), (13, 8, 1, 1), (13, 10, 2, 1), (14, 3, 1, 2), (14, 4, 2, 2), (12, 24, 8, 2), (14, 8, 1, 4),
                                                 (14, 10, 2, 4), (15, 2, 1, 4), (15, 2, 1, 5), (15, 10, 2, 2),
                                                 (16, 3, 1, 4), (16, 3, 1, 5), (15, 3, 1, 3), (15, 8, 1, 2)])
def test_encryption_of_a_mixed_chain(oracle, capi, logn, L, size_p, items):
    """Encryption's blocks pass deals the limbs' workgroups to all XCDs for up to four items, from 3 workgroups for two CUs on, with limbs
    of 2^14 words and less from 3 a CU for two items and from 12 for more; with one special prime limbs of 2^16 words, up to 16 of 2^15 and
    single encryptions, but not four items of few limbs; its ModDown from 3 a CU on for one item or limbs of 2^15."""
    bits = [60] + [40] * (L - 1) + [60] * size_p
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, size_p)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    key = oracle.chacha_key(3)
    kp = key.ctypes.data_as(C.POINTER(C.c_uint32))
    rng = np.random.default_rng(logn + L)
    pk, plain = rand_limbs(p, rng, range(p.size_qp), n_polys=2), rand_limbs(p, rng, range(p.size_q), n_polys=items)
    cts = np.zeros((items, 2, L, n), dtype=np.uint64)
    cts[:, 0] = plain
    dpk, dcts = DeviceArray(capi, host=pk), DeviceArray(capi, host=cts)
    ws = DeviceArray(capi, shape=(lib.he_encrypt_batch_workspace_words(h, L, items),))
    capi.check(lib.he_encrypt_batch(h, L, items, dpk.ptr, kp, 11, dcts.ptr, ws.ptr, None))
    got = dcts.numpy()
    for k in sorted({0, items - 1}):
        u = p.ntt_fwd(p.sample_ternary(key, 11 + 3 * k, p.size_qp))
        for i in range(2):
            e = p.ntt_fwd(p.sample_error(key, 12 + 3 * k + i, p.size_qp))
            want = p.moddown(np.ascontiguousarray(p.mul_add(u, pk[i], e)))
            assert (got[k, i] == (p.add(want, plain[k]) if i == 0 else want)).all(), (k, i)


@pytest.mark.parametrize("logn,L,polys", [(16, 3, 2), (16, 4, 2), (16, 5, 2), (16, 3, 4), (15, 6, 4)])
def test_moddown_and_rescale_of_a_mixed_chain(oracle, capi, logn, L, polys):
    """Their epilogue's workgroups, 768 and more, go to all XCDs for up to eight limbs of two polynomials."""
    cahel, parms, ctx, p = make_pair(oracle, logn, [60] + [40] * (L - 1) + [60], 1)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    cx = rand_limbs(p, np.random.default_rng(L + polys), range(L + 1), n_polys=polys)
    dcx, dct, ws = DeviceArray(capi, host=cx), DeviceArray(capi, host=cx[:, :L]), DeviceArray(capi, shape=(polys, L, n))
    down, low = DeviceArray(capi, shape=(polys, L, n)), DeviceArray(capi, shape=(polys, L - 1, n))
    capi.check(lib.he_moddown(h, L, dcx.ptr, down.ptr, polys, 0, ws.ptr, None))
    capi.check(lib.he_rescale(h, dct.ptr, low.ptr, polys, L, ws.ptr, None))
    assert (down.numpy() == np.stack([p.moddown(x) for x in cx])).all()
    assert (low.numpy() == p.rescale(np.ascontiguousarray(cx[:, :L]))).all()


@pytest.mark.parametrize("bits", [[50] * 20, [60] + [40] * 15 + [60] * 4])
@pytest.mark.parametrize("L", [15, 16])
def test_modup_on_both_sides_of_the_twiddles_worked_out(oracle, capi, bits, L):
    """FP64: 61 and 64 transformed limbs of 2^16 words.  Both arithmetics work them out from 36 on."""
    cahel, parms, ctx, p = make_pair(oracle, 16, bits, 4)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    c = rand_limbs(p, np.random.default_rng(L), range(L))
    for i in range(0, L, 3):
        c[i] = p.moduli[i] - 1
    dc, dy, ws = DeviceArray(capi, host=c), DeviceArray(capi, shape=(4, L + 4, n)), DeviceArray(capi, shape=(2 * L, n))
    capi.check(lib.he_modup(h, L, dc.ptr, dy.ptr, ws.ptr, None))
    assert (dy.numpy() == p.modup(c)).all()


@pytest.mark.parametrize("bits", [[50] * 17, [50, 49, 30] * 5 + [50, 49], [60] + [40] * 15 + [60]])
@pytest.mark.parametrize("L", [15, 16])
def test_epilogues_on_both_sides_of_the_twiddles_worked_out(oracle, capi, bits, L):
    """FP64: 1024 waves at 256 CUs, ModDown of 16 limbs of 2^13 words; the rescale has a limb less.  Words of q - 1 throughout, and random ones."""
    cahel, parms, ctx, p = make_pair(oracle, 13, bits, 1)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    tables = list(range(L)) + [p.size_q]
    cx = rand_limbs(p, np.random.default_rng(L), tables, n_polys=2)
    for i, t in enumerate(tables):
        cx[1, i] = p.moduli[t] - 1
    dcx, dct, ws = DeviceArray(capi, host=cx), DeviceArray(capi, host=cx[:, :L]), DeviceArray(capi, shape=(2, L, n))
    down, low = DeviceArray(capi, shape=(2, L, n)), DeviceArray(capi, shape=(2, L - 1, n))
    capi.check(lib.he_moddown(h, L, dcx.ptr, down.ptr, 2, 0, ws.ptr, None))
    capi.check(lib.he_rescale(h, dct.ptr, low.ptr, 2, L, ws.ptr, None))
    assert (down.numpy() == np.stack([p.moddown(x) for x in cx])).all()
    assert (low.numpy() == p.rescale(np.ascontiguousarray(cx[:, :L]))).all()


@pytest.mark.parametrize("chain", sorted(CHAINS))
@pytest.mark.parametrize("logn,L,items", [(12, 8, 19), (12, 8, 20), (13, 5, 16), (15, 2, 5), (15, 2, 6)])
def test_products_on_both_sides_of_the_dealt_tensor_product(oracle, capi, chain, logn, L, items):
    """A batch's tensor product deals its workgroups to all XCDs from 10 * 2^16 words a polynomial on, from 6 * 2^16 with limbs of 2^15."""
    bits = (CHAINS[chain] * 2)[:L + 1]
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, 1)
    rng = np.random.default_rng(logn + items)
    lib, h = capi.lib(), ctx.he_handle()
    host = [rand_limbs(p, rng, range(p.size_qp), n_polys=2) for _ in range(2)]
    dev = [DeviceArray(capi, host=k) for k in host]
    keys = capi.evk_array([dev[d % 2].ptr for d in range(L)])
    a, b = (rand_limbs(p, rng, range(L), n_polys=2 * items).reshape(items, 2, L, p.n) for _ in range(2))
    da, db, out = DeviceArray(capi, host=a), DeviceArray(capi, host=b), DeviceArray(capi, shape=(items, 2, L - 1, p.n))
    ws = DeviceArray(capi, shape=(lib.he_multiply_relin_rescale_batch_workspace_words(h, L, items),))
    capi.check(lib.he_multiply_relin_rescale_batch(h, L, items, da.ptr, db.ptr, keys, out.ptr, ws.ptr, None))
    got = out.numpy()
    for k in (0, items // 2, items - 1):
        d = p.tensor(a[k], b[k])
        ks = p.key_switch(d[2], [host[j % 2] for j in range(L)])
        assert (got[k] == p.rescale(np.stack([p.add(d[i], ks[i]) for i in range(2)]))).all(), k
