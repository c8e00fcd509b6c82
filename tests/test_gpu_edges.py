"""Calls at the ends of what the entry points take: more rows of sums than one launch or one call of the C-ABI holds, decryption at
the key level, batches of more threads than a launch has, plaintexts used on another lane while their encoding runs, buffers that are aligned to one
word only."""
import ctypes as C

import numpy as np
import pytest

import test_gpu_fused_rows as fused_rows
import test_gpu_passes as passes
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


def test_products_refuse_the_scales_that_multiply_refuses(oracle):
    """90 bits of modulus at this level: a product of scale 2^89 is one, of scale 2^90 none."""
    cahel, parms, ctx, p = make_pair(oracle, 9, [50, 40, 50], 1)
    sk, pk = keys_for(cahel, parms, ctx)
    ct = pk.encrypt_asymmetric(ctx, cahel.ckks_encoder(ctx).encode(ctx, np.ones(p.n // 2), 2.0 ** 20))
    for log_scale in (44.5, 45.0, 60.0):
        ct.set_scale(2.0 ** log_scale)
        calls = [lambda: cahel.multiply(ctx, ct, ct, cahel.ciphertext(ctx)), lambda: cahel.multiply_sum(ctx, [[ct, ct]], [ct, ct])]
        for call in calls:
            if log_scale < 45:
                call()
            else:
                with pytest.raises(ValueError, match="scale out of bounds"):
                    call()


def test_encodings_used_on_other_lanes_at_once(oracle, capi):
    """encode returns while its lane works: what another lane, another stream or a copy reads is the whole plaintext."""
    cahel, parms, ctx, p = make_pair(oracle, 16, [60, 40, 40, 60], 1)
    sk, pk = keys_for(cahel, parms, ctx)
    sk.set_noise_flooding(False)
    enc, rng, lib = cahel.ckks_encoder(ctx), np.random.default_rng(3), capi.lib()
    z = rng.uniform(-1, 1, (6, p.n // 2))
    want = [enc.encode(ctx, row, 2.0 ** 40).to_numpy() for row in z]
    cahel._synchronize()
    other = C.c_void_p()
    capi.check(lib.he_stream_create(C.byref(other)))
    try:
        for turn, lane in enumerate([1, 2, 0, 3]):
            cahel._set_lane(0)
            plains = [enc.encode(ctx, row, 2.0 ** 40) for row in z]
            words = np.empty_like(want[5])
            capi.check(lib.he_memcpy_d2h(words.ctypes.data, plains[5].data_ptr(), words.nbytes, other))
            cahel._set_lane(lane)
            got = plains[4].to_numpy()
            cts = [pk.encrypt_asymmetric(ctx, plain) for plain in plains[:4]]
            back = [enc.decode_array(ctx, sk.decrypt(ctx, ct)) for ct in cts]
            assert (words == want[5]).all() and (got == want[4]).all(), (turn, lane)
            assert all(np.abs(b - row).max() < 1e-5 for b, row in zip(back, z)), (turn, lane)
            cahel._synchronize()
    finally:
        cahel._set_lane(0)
        lib.he_stream_destroy(other)


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


@pytest.mark.parametrize("logn,bits,size_p", [(9, [50, 49, 50], 1), (12, [60, 40, 40, 50, 60, 60], 2), (13, [60, 58, 60], 1)])
def test_decryption_at_the_key_level(oracle, capi, logn, bits, size_p):
    """A ciphertext over all primes, the special ones among them: encrypted and decrypted through pyCAHEL, and he_decrypt_flood of 2 and
    3 polynomials."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, size_p)
    sk, pk = keys_for(cahel, parms, ctx)
    enc = cahel.ckks_encoder(ctx)
    plain = enc.encode_to(ctx, np.linspace(-1, 1, p.n // 2), 0, 2.0 ** 30)
    ct = pk.encrypt_asymmetric(ctx, plain)
    assert ct.chain_index() == 0 and ct.coeff_modulus_size() == p.size_qp
    got = sk.decrypt(ctx, ct)
    assert got.chain_index() == 0
    # the difference of the decryption and the plaintext: encryption's and flooding's noise, the same small integers modulo every prime
    diff = p.ntt_inv(np.ascontiguousarray(p.sub(got.to_numpy(), plain.to_numpy())))
    signed = [np.where(d > np.uint64(q // 2), d.astype(np.int64) - q, d.astype(np.int64)) for d, q in zip(diff, p.moduli)]
    assert all((s == signed[0]).all() for s in signed) and 0 < np.abs(signed[0]).max() < 2 ** 20
    lib, h, rng = capi.lib(), ctx.he_handle(), np.random.default_rng(logn)
    key, cdt = oracle.chacha_key(3), oracle.gauss_cdt()
    kp = key.ctypes.data_as(C.POINTER(C.c_uint32))
    for limbs in (p.size_q, p.size_qp):
        ct3, s = (rand_limbs(p, rng, range(limbs), n_polys=k) for k in (3, 2))
        dct, dsk, dcdt = DeviceArray(capi, host=ct3), DeviceArray(capi, host=s), DeviceArray(capi, host=cdt)
        out, noise = DeviceArray(capi, shape=(limbs, p.n)), DeviceArray(capi, shape=(p.n // 8,))
        e = p.ntt_fwd(p.sample_gauss(key, 5, limbs, cdt))
        for size in (2, 3):
            capi.check(lib.he_decrypt_flood(h, dct.ptr, size, limbs, dsk.ptr, limbs * p.n, kp, 5, dcdt.ptr, len(cdt), out.ptr, noise.ptr, None))
            want = p.mul_add(ct3[1], s[0], ct3[0])
            want = p.mul_add(ct3[2], s[1], want) if size == 3 else want
            assert (out.numpy() == p.add(want, e)).all(), (limbs, size)
    assert lib.he_decrypt_flood(h, dct.ptr, 2, p.size_qp + 1, dsk.ptr, 0, kp, 5, dcdt.ptr, len(cdt), out.ptr, noise.ptr, None) == -1


def allocate(capi, words):
    """words of device memory, zero; skips where the card has no room for them."""
    ptr = C.c_void_p()
    if capi.lib().he_malloc(C.byref(ptr), 8 * words) != 0:
        pytest.skip("not enough free device memory")
    capi.check(capi.lib().he_memset_zero(ptr.value, 8 * words, None))
    return ptr.value


@pytest.mark.parametrize("logn,bits", [(16, [50, 50]), (16, [60, 60]), (16, [60, 40, 60]), (10, [50, 50]), (10, [60, 40, 60]),
                                       (12, [50, 50]), (12, [60, 60]), (12, [60, 40, 60])])
def test_transforms_of_more_words_than_a_launch_holds(oracle, capi, logn, bits):
    """2^34 words (137 GB) and some: a thread of the rows pass, or of a whole limb of 2^10 or 2^12 words, takes four (16 at 2^12, 50
    bits), and a launch has fewer than 2^32 threads."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, 1)
    lib, h, n, limbs = capi.lib(), ctx.he_handle(), p.n, len(bits) - 1
    polys, rng = ((1 << (34 - logn)) + 8) // limbs, np.random.default_rng(limbs)
    data = allocate(capi, polys * limbs * n)
    try:
        last = 0xffffffff // (n // 4) // limbs       # the polynomials of the first launch
        xs = {k: rand_limbs(p, rng, range(limbs)) for k in (0, 8, last - 1, last, last + 1, polys - 1)}
        at = lambda k: data + 8 * k * limbs * n
        for k, x in xs.items():
            capi.check(lib.he_memcpy_h2d(at(k), x.ctypes.data, x.nbytes, None))
        for transform, want in ((lib.he_ntt_forward, {k: p.ntt_fwd(x.copy()) for k, x in xs.items()}), (lib.he_ntt_inverse, xs)):
            capi.check(transform(h, data, polys, limbs, limbs, 0, limbs, 0, None))
            got = np.empty((limbs, n), dtype=np.uint64)
            for k in xs:
                capi.check(lib.he_memcpy_d2h(got.ctypes.data, at(k), got.nbytes, None))
                assert (got == want[k]).all(), k
    finally:
        lib.he_free(data)


def test_encryptions_of_more_words_than_a_launch_holds(oracle, capi):
    """he_encrypt_batch of 8192 items over 11 limbs of 2^16 words (193 GB): its passes have more than 2^32 threads."""
    cahel, parms, ctx, p = make_pair(oracle, 16, [50] * 16, 8)
    lib, h, n, L, items = capi.lib(), ctx.he_handle(), p.n, 3, 8192
    pk = DeviceArray(capi, host=rand_limbs(p, np.random.default_rng(1), range(p.size_qp), n_polys=2))
    kp = oracle.chacha_key(3).ctypes.data_as(C.POINTER(C.c_uint32))
    cts = allocate(capi, items * 2 * L * n)
    try:
        ws = allocate(capi, lib.he_encrypt_batch_workspace_words(h, L, items))
        try:
            capi.check(lib.he_encrypt_batch(h, L, items, pk.ptr, kp, 7, cts, ws, None))
            zero, one = DeviceArray(capi, host=np.zeros((L, n), dtype=np.uint64)), DeviceArray(capi, shape=(2, L, n))
            got = np.empty((2, L, n), dtype=np.uint64)
            first = 0xffffffff // 192 // (11 * 256)    # the items of the first launch
            for k in (0, first // 2, first - 1, first, items - 1):
                capi.check(lib.he_encrypt(h, L, zero.ptr, pk.ptr, kp, 7 + 3 * k, one.ptr, ws, None))
                capi.check(lib.he_memcpy_d2h(got.ctypes.data, cts + 16 * k * L * n, got.nbytes, None))
                assert (got == one.numpy()).all(), k
        finally:
            lib.he_free(ws)
    finally:
        lib.he_free(cts)


@pytest.mark.parametrize("first,count", [(4, 1), (3, 2), (0, 5), (2 ** 32 - 1, 1), (2 ** 32 - 1, 4), (2 ** 32 - 2, 3), (2, 2 ** 32 - 1)])
def test_limbs_past_the_last_prime_are_refused(oracle, capi, first, count):
    """Runs of limbs that end behind the last of four primes, and runs whose end is beyond 2^32: refused before anything is launched."""
    cahel, parms, ctx, p = make_pair(oracle, 9, [50, 40, 40, 50], 1)
    lib, h = capi.lib(), ctx.he_handle()
    a, b, out = (DeviceArray(capi, host=np.zeros((8, p.n), dtype=np.uint64)) for _ in range(3))
    kp = oracle.chacha_key(3).ctypes.data_as(C.POINTER(C.c_uint32))
    calls = [lib.he_add(h, a.ptr, b.ptr, out.ptr, 1, count, first, None), lib.he_negate(h, a.ptr, out.ptr, 1, count, first, None),
             lib.he_multiply_add(h, a.ptr, b.ptr, a.ptr, out.ptr, 1, count, first, 0, None),
             lib.he_add_p_multiple(h, a.ptr, b.ptr, out.ptr, first, count, None), lib.he_decompose_real(h, a.ptr, out.ptr, count, first, None)]
    for transform in (lib.he_ntt_forward, lib.he_ntt_inverse):
        calls.append(transform(h, out.ptr, 1, count, count, first, count, 0, None))
        calls.append(transform(h, out.ptr, 1, count, count, 0, 0, first, None))
    calls.append(lib.he_sample(h, 0, kp, 1, out.ptr, count, first, count, 0, None, 0, None))
    assert calls == [-1] * len(calls)


@pytest.mark.parametrize("bits,size_p", [([50, 40, 40, 50], 1), ([50, 40, 40, 40, 50, 50], 2), ([60, 40, 40, 40, 60, 60], 2)])
@pytest.mark.parametrize("logn", [9, 12])
def test_moddown_of_no_polynomials(oracle, capi, logn, bits, size_p):
    """Nothing to do, with any number of special primes (the number is a divisor where the conversions are batched)."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, size_p)
    words = np.full((p.size_qp, p.n), 7, dtype=np.uint64)
    cx, out, ws = (DeviceArray(capi, host=words) for _ in range(3))
    for add in (0, 1):
        assert capi.lib().he_moddown(ctx.he_handle(), p.size_q, cx.ptr, out.ptr, 0, add, ws.ptr, None) == 0
    assert all((a.numpy() == words).all() for a in (cx, out, ws))


class OddArray(DeviceArray):
    """A device buffer that starts 8 bytes behind a 16-byte boundary."""

    def __init__(self, capi, shape=None, host=None, dtype=np.uint64):
        host = None if host is None else np.ascontiguousarray(host)
        self.capi = capi
        self.shape, self.dtype = (tuple(shape), np.dtype(dtype)) if host is None else (host.shape, host.dtype)
        self.nbytes = int(np.prod(self.shape)) * self.dtype.itemsize
        self.base = C.c_void_p()
        capi.check(capi.lib().he_malloc(C.byref(self.base), self.nbytes + 16), "he_malloc")
        self.ptr = self.base.value + 8
        assert self.ptr % 16 == 8
        if host is not None:
            capi.check(capi.lib().he_memcpy_h2d(self.ptr, host.ctypes.data, self.nbytes, None), "h2d")

    def free(self):
        if self.ptr:
            self.capi.lib().he_free(self.base.value)
            self.ptr = None


@pytest.mark.parametrize("chain", ["fp", "int", "mixed"])
def test_buffers_aligned_to_one_word(oracle, capi, monkeypatch, chain):
    """The header asks for 8-byte alignment; the passes and what is fused with them move 16 bytes at a time."""
    monkeypatch.setattr(passes, "DeviceArray", OddArray)
    passes.test_batched_transforms(oracle, capi, chain, 15, 5, 30)
    passes.test_batched_transforms(oracle, capi, chain, 12, 3, 2)
    passes.test_encrypt_and_decrypt(oracle, capi, chain, 13, 2, 3)
    passes.test_bounded_encoding_and_real_decoding(oracle, capi, chain, 13, 4096, 3)
    passes.test_hoisting_of_one_ciphertext(oracle, capi, chain, 12, 2, 4, 3)
    passes.test_hoisting_of_one_ciphertext(oracle, capi, chain, 16, 2, 4, 3)
    for local in (False, True):
        passes.test_hoisting_of_batches(oracle, capi, chain, local, 12, 2, 4, 4, 5)
    passes.test_sums_of_ciphertexts_and_products(oracle, capi, chain, 13, 2, 2, 17)


@pytest.mark.parametrize("case", [c for c in fused_rows.CASES if c[0] in (12, 14)] + [(16, [50] * 6, 2, (4,))])
def test_key_switches_of_buffers_aligned_to_one_word(oracle, capi, monkeypatch, case):
    monkeypatch.setattr(fused_rows, "DeviceArray", OddArray)
    fused_rows.test_entry_points_with_fused_conversion(oracle, capi, monkeypatch, *case, "0")
    fused_rows.test_multiply_relin_rescale_entry_point(oracle, capi, monkeypatch, *case, "0")
    for inner in ("fused", "fp_kernel"):
        fused_rows.test_multiply_relin_rescale_batch_equals_single_calls(oracle, capi, monkeypatch, *case[:3], case[3][0], 3, inner)
