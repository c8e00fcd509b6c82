"""What only a caller of the C-ABI can ask for: primes of 61 bits, the largest that he_context_create takes (the host layer stops at
60), where the lazy sums of the integer kernels are relieved more often or have less room; and chains of more than 64 primes, whose
limbs past the 64th no mask of back ends covers.  The cases of test_gpu_passes and key switches with operands that are q - 1 in many
places, against the oracle, which also supplies the tables."""
import ctypes as C

import numpy as np
import pytest

import test_gpu_passes as passes
from gpu_util import DeviceArray, rand_limbs

pytestmark = pytest.mark.gpu


class ContextDesc(C.Structure):
    _fields_ = [(f, C.c_uint32) for f in ("log_n", "size_q", "size_p", "reserved")] + \
               [(f, C.c_void_p) for f in ("moduli", "barrett", "psi", "ipsi_div2", "p_mod_q", "pinv_mod_q", "phat_inv_mod_p", "phat_mod_q")]


class LevelDesc(C.Structure):
    _fields_ = [("L", C.c_uint32), ("beta", C.c_uint32)] + [(f, C.c_void_p) for f in ("part_hat_inv", "digit_mats", "digit_mat_off", "qlast_inv")]


class Context:
    """A device context over the oracle's tables."""

    def __init__(self, capi, p):
        self.lib, self.handle = capi.lib(), C.c_void_p()
        pairs = lambda w, q: np.stack([w, np.array([(int(x) << 64) // int(m) for x, m in zip(w, q)], dtype=np.uint64)], axis=-1)
        q, special = p.mod[:p.size_q], p.mod[p.size_q:]
        host = [p.mod, p.ratio, np.stack([p.tw, p.twq], axis=-1), np.stack([p.itw, p.itwq], axis=-1), pairs(p.p_mod_q, q),
                pairs(p.pinv_mod_q, q), pairs(p.phat_inv, special), p.mat_p2q]
        host = [np.ascontiguousarray(x) for x in host]
        capi.check(self.lib.he_context_create(C.byref(ContextDesc(p.logn, p.size_q, p.size_p, 0, *[x.ctypes.data for x in host])), C.byref(self.handle)))
        for L in range(1, p.size_q + 1):
            lt = p.level(L)
            host = [np.ascontiguousarray(x) for x in (pairs(lt.hatinv, q), lt.mats, lt.mat_off, pairs(lt.qlast_inv, q))]
            capi.check(self.lib.he_context_set_level(self.handle, C.byref(LevelDesc(L, lt.beta, *[x.ctypes.data for x in host]))))

    def he_handle(self):
        return self.handle.value

    def __del__(self):
        if self.handle:
            self.lib.he_context_destroy(self.handle)


def make_pair(oracle, logn, bits, size_p):
    """gpu_util.make_pair without the host layer: (None, None, context, oracle Params)."""
    import lancelot_amd  # noqa: F401
    import pyCAHEL as cahel
    from lancelot_amd import capi
    pools = {b: list(cahel._get_primes(1 << logn, b, bits.count(b))) for b in set(bits)}
    values = [int(pools[b].pop(0)) for b in bits]
    assert all(v >> 60 for v, b in zip(values, bits) if b == 61)
    p = oracle.Params(logn, values, size_p)
    return None, None, Context(capi, p), p


@pytest.fixture(scope="module")
def capi():
    from lancelot_amd import capi as c
    c.lib()
    return c


@pytest.fixture
def cases(monkeypatch):
    monkeypatch.setattr(passes, "make_pair", make_pair)
    monkeypatch.setitem(passes.CHAINS, "all", [61] * 6)
    monkeypatch.setitem(passes.CHAINS, "some", [61, 40, 61, 50, 61, 61])
    return passes


@pytest.mark.parametrize("chain", ["all", "some"])
@pytest.mark.parametrize("logn", [9, 12, 14, 16])
def test_transforms_encryption_and_sums(oracle, capi, cases, chain, logn):
    cases.test_batched_transforms(oracle, capi, chain, logn, 4, 7)
    cases.test_encrypt_and_decrypt(oracle, capi, chain, logn, 1, 3)
    for count in (1, 16, 33):
        cases.test_sums_of_ciphertexts_and_products(oracle, capi, chain, logn, 2, 2, count)


@pytest.mark.parametrize("chain", ["all", "some"])
@pytest.mark.parametrize("logn,size_p,L,n_steps,items", [(9, 1, 4, 16, 5), (10, 2, 4, 3, 2), (12, 1, 3, 21, 1), (16, 1, 2, 15, 4)])
def test_hoisting(oracle, capi, cases, chain, logn, size_p, L, n_steps, items):
    if items == 1:
        cases.test_hoisting_of_one_ciphertext(oracle, capi, chain, logn, size_p, L, n_steps)
    else:
        for local in (False, True):
            cases.test_hoisting_of_batches(oracle, capi, chain, local, logn, size_p, L, n_steps, items)


@pytest.mark.parametrize("logn,bits,size_p,levels", [(12, [61] * 16, 8, (8, 3)), (13, [61, 40, 61, 61, 50, 61, 61, 61], 4, (4, 3)),
                                                     (16, [61] * 6, 2, (4, 3))])
def test_fused_conversions(oracle, capi, cases, logn, bits, size_p, levels):
    cases.test_conversion_fused_on_integers(oracle, capi, logn, bits, size_p, levels)


@pytest.mark.parametrize("logn,bits,size_p,L,items", [
    (9, [61] * 18, 9, 9, 1), (11, [61] * 9, 1, 8, 1), (11, [61] * 9, 1, 8, 5), (14, [61, 40, 61, 61], 1, 3, 1), (14, [61, 40, 61, 61], 1, 3, 3),
    (15, [61] * 6, 2, 4, 1), (15, [61] * 6, 2, 4, 5), (12, [50] * 70, 2, 68, 1), (12, [50] * 70, 2, 66, 2), (11, [60, 50] * 36, 3, 67, 1),
    (10, [40] * 65, 1, 64, 4)])
def test_products_of_largest_residues(oracle, capi, logn, bits, size_p, L, items):
    """he_multiply_relin_rescale of ciphertexts whose words are mostly q - 1, with a key whose words all are, single and as a batch;
    he_rotate and a hoisted sum of as many products as a launch takes."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, size_p)
    lib, h, n = capi.lib(), ctx.he_handle(), p.n
    top = np.array(p.moduli, dtype=np.uint64)[:, None] - np.uint64(1)
    key = np.ascontiguousarray(np.broadcast_to(top, (2, p.size_qp, n)))
    ct = np.ascontiguousarray(np.broadcast_to(top[:L], (2, L, n)))
    ct[1, :, ::3] = rand_limbs(p, np.random.default_rng(L), range(L))[:, ::3]
    beta = -(-L // size_p)
    dkey, dct = DeviceArray(capi, host=key), DeviceArray(capi, host=np.stack([ct] * items))
    evk = capi.evk_array([dkey.ptr] * beta)
    ws = DeviceArray(capi, shape=(max(lib.he_multiply_relin_rescale_batch_workspace_words(h, L, items),
                                      lib.he_multiply_relin_rescale_workspace_words(h, L)),))
    out = DeviceArray(capi, shape=(items, 2, L - 1, n))
    if items == 1:
        capi.check(lib.he_multiply_relin_rescale(h, L, dct.ptr, dct.ptr, evk, out.ptr, ws.ptr, None))
    else:
        capi.check(lib.he_multiply_relin_rescale_batch(h, L, items, dct.ptr, dct.ptr, evk, out.ptr, ws.ptr, None))
    want = p.rescale(p.relinearize(p.tensor(ct, ct), [key] * beta))
    assert all((got == want).all() for got in out.numpy())
    rot = DeviceArray(capi, shape=(items, 2, L, n))
    n_steps = 64 // beta
    elts = [pow(5, k + 1, 2 * n) for k in range(n_steps)]
    flat, d_elts = capi.evk_array([dkey.ptr] * (beta * n_steps)), (C.c_uint32 * n_steps)(*elts)
    capi.check(lib.he_hoisted_rotations_batch(h, L, items, dct.ptr, flat, d_elts, n_steps, 0, rot.ptr, ws.ptr, None))
    want = p.hoisting(ct, elts, [[key] * beta] * n_steps)
    assert all((got == want).all() for got in rot.numpy())
    if items == 1:
        capi.check(lib.he_rotate(h, L, dct.ptr, evk, rot.ptr, 5, ws.ptr, None))
        assert (rot.numpy()[0] == p.apply_galois(ct, 5, [key] * beta)).all()


@pytest.mark.parametrize("logn,bits", [(12, [50] * 68), (12, [60, 50] * 34), (13, [61] * 68)])
def test_encryption_and_decoding_of_long_chains(oracle, capi, logn, bits):
    """More than 64 primes: encryption and decryption over all data limbs, and the decoding of a few."""
    cahel, parms, ctx, p = make_pair(oracle, logn, bits, 2)
    lib, h, n, L = capi.lib(), ctx.he_handle(), p.n, p.size_q
    rng, key, cdt = np.random.default_rng(logn), oracle.chacha_key(3), oracle.gauss_cdt()
    kp = key.ctypes.data_as(C.POINTER(C.c_uint32))
    pk, plain = rand_limbs(p, rng, range(p.size_qp), n_polys=2), rand_limbs(p, rng, range(L))
    dpk, dplain, dct = DeviceArray(capi, host=pk), DeviceArray(capi, host=plain), DeviceArray(capi, shape=(2, L, n))
    ws = DeviceArray(capi, shape=(lib.he_encrypt_batch_workspace_words(h, L, 1),))
    capi.check(lib.he_encrypt(h, L, dplain.ptr, dpk.ptr, kp, 11, dct.ptr, ws.ptr, None))
    got, u = dct.numpy(), p.ntt_fwd(p.sample_ternary(key, 11, p.size_qp))
    for i in range(2):
        e = p.ntt_fwd(p.sample_error(key, 12 + i, p.size_qp))
        want = p.moddown(np.ascontiguousarray(p.mul_add(u, pk[i], e)))
        assert (got[i] == (p.add(want, plain) if i == 0 else want)).all(), i
    sk = rand_limbs(p, rng, range(p.size_qp))
    dsk, dcdt, out, noise = DeviceArray(capi, host=sk), DeviceArray(capi, host=cdt), DeviceArray(capi, shape=(L, n)), DeviceArray(capi, shape=(n // 8,))
    capi.check(lib.he_decrypt_flood(h, dct.ptr, 2, L, dsk.ptr, 0, kp, 5, dcdt.ptr, len(cdt), out.ptr, noise.ptr, None))
    want = p.add(p.mul_add(got[1], np.ascontiguousarray(sk[:L]), got[0]), p.ntt_fwd(p.sample_gauss(key, 5, L, cdt)))
    assert (out.numpy() == want).all()
    slots, scale = n // 2, 2.0 ** 40
    for limbs in (2, 5, 64):
        z = rng.uniform(-1, 1, slots)
        re, enc = DeviceArray(capi, host=z), DeviceArray(capi, shape=(limbs, n))
        ews = DeviceArray(capi, shape=(lib.he_ckks_encode_batch_workspace_words(h, 1),))
        capi.check(lib.he_ckks_encode_bounded(h, re.ptr, None, slots, slots, scale, limbs, 1, slots, enc.ptr, limbs, ews.ptr, None))
        real, rws = DeviceArray(capi, shape=(slots,), dtype=np.float64), DeviceArray(capi, shape=(lib.he_ckks_decode_real_workspace_words(h, limbs, slots),))
        capi.check(lib.he_ckks_decode_real(h, enc.ptr, limbs, slots, scale, real.ptr, slots, rws.ptr, None))
        assert np.abs(real.numpy() - z).max() < 2.0 ** -25, limbs
