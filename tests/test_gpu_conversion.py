"""ModUp and ModDown's basis conversions on the matrix units, bit-exact
against the oracle: every source count of a four-source step (1 .. 16),
targets that do and do not fill a group of four, a batch of lines, moduli at
both ends of the fused range (just above 2^33, just below 2^60) and inputs of
extreme residues; and the small rings' conversions inside the transforms up
to, and past, their eight sources."""
import numpy as np
import pytest

import oracle as O
from gpu_helpers import edge_patterns, residues

pytestmark = pytest.mark.gpu
F = pytest.importorskip("fhemamba_amd")

# (log_n, Q limbs, bits of Q, P limbs, bits of P, dnum): alpha = ceil(L / dnum)
SHAPES = [(13, 1, 59, 1, 60, 1), (13, 6, 59, 3, 60, 2), (13, 13, 34, 5, 60, 3),
          (13, 16, 60, 16, 60, 1), (14, 15, 50, 15, 59, 1), (15, 9, 59, 4, 60, 2),
          (16, 11, 59, 7, 60, 2), (17, 10, 60, 6, 60, 2),
          (12, 8, 59, 8, 60, 1), (12, 9, 59, 9, 60, 1), (10, 5, 45, 2, 60, 3),
          (6, 4, 30, 2, 40, 4)]


@pytest.mark.parametrize("log_n,L,qbits,K,pbits,dnum", SHAPES)
def test_key_switch_bit_exact(log_n, L, qbits, K, pbits, dnum):
    q = O.ntt_friendly_primes(log_n, qbits, L)
    p = O.ntt_friendly_primes(log_n, pbits, K, skip=q)
    ctx, orc = F.Context(log_n, q, p, dnum, sampling="seeded"), O.Ctx(log_n, q, p, dnum)
    rng = np.random.default_rng(17)
    key = residues(rng, list(q) + list(p), (ctx.dnum, 2), ctx.n)
    dkey = ctx.load_key(key)
    for nq in sorted({1, (L + 1) // 2, max(1, L - 1), L}):
        a = residues(rng, q[:nq], (1,), ctx.n)
        assert np.array_equal(ctx.keyswitch(ctx.upload(a), dkey).numpy(),
                              orc.keyswitch(a[0], key)), nq
    for pat in edge_patterns(q[:L], ctx.n):
        assert np.array_equal(ctx.keyswitch(ctx.upload(pat[None]), dkey).numpy(),
                              orc.keyswitch(pat, key))
    ct3 = [residues(rng, q, (3,), ctx.n) for _ in range(3)]
    outs = ctx.relinearize_many([ctx.upload(c) for c in ct3], dkey)
    for c, o in zip(ct3, outs):
        assert np.array_equal(o.numpy(), orc.relinearize(c, key))
    if L > 1:
        many = ctx.rescale_many([ctx.upload(c) for c in ct3])
        for c, o in zip(ct3, many):
            assert np.array_equal(o.numpy(), orc.rescale(c))
    ctx.close()


# (log_n, Q limbs, P limbs, dnum, key switches): the middle kernel's workgroups
# of 4 waves (lines that fill no more; batches whose 4-wave form keeps at least
# as many waves on a compute unit), 8 and 16, one batch of targets and several,
# whole and ragged ones.
FORMS = [(13, 3, 1, 3, 12), (13, 12, 5, 2, 16), (13, 12, 5, 2, 2), (14, 11, 9, 1, 8),
         (15, 9, 4, 2, 8), (16, 9, 3, 2, 2), (16, 9, 9, 1, 2), (17, 6, 1, 6, 1), (17, 9, 5, 2, 1),
         (17, 9, 5, 2, 2), (17, 13, 12, 1, 1)]


@pytest.mark.parametrize("log_n,L,K,dnum,count", FORMS)
def test_middle_kernel_workgroup_forms(log_n, L, K, dnum, count):
    q = O.ntt_friendly_primes(log_n, 59, L)
    p = O.ntt_friendly_primes(log_n, 60, K, skip=q)
    ctx, orc = F.Context(log_n, q, p, dnum, sampling="seeded"), O.Ctx(log_n, q, p, dnum)
    rng = np.random.default_rng(23)
    key = residues(rng, list(q) + list(p), (ctx.dnum, 2), ctx.n)
    dkey = ctx.load_key(key)
    ct3 = [residues(rng, q, (3,), ctx.n) for _ in range(min(2, count))]
    want = [orc.relinearize(c, key) for c in ct3]
    outs = ctx.relinearize_many([ctx.upload(ct3[r % 2]) for r in range(count)], dkey)
    for r, o in enumerate(outs):
        assert np.array_equal(o.numpy(), want[r % 2]), r
    gal = [5, 2 * ctx.n - 1]
    ct = ctx.upload(ct3[0][:2])
    want = [orc.rotate(ct3[0][:2], key, g) for g in gal]
    outs = ctx.rotate_hoisted(ct, ctx.rotation_precompute(ct), [dkey] * count,
                              [gal[r % 2] for r in range(count)])
    for r, o in enumerate(outs):
        assert np.array_equal(o.numpy(), want[r % 2]), r
    ctx.close()


# Q bit sizes, last limb dropped first: primes of one chain, a last prime many
# times (reduced after its lift) and too many times (four launches) the others.
RESCALES = [(13, (59, 59, 59)), (14, (60, 45, 59)), (15, (60, 34, 60)), (16, (45, 59)),
            (17, (60, 59, 59)), (11, (60, 40, 59)), (13, (61, 59, 59))]


@pytest.mark.parametrize("log_n,bits", RESCALES)
def test_rescale_moduli(log_n, bits):
    q = []
    for b in bits:
        q += O.ntt_friendly_primes(log_n, b, 1, skip=q)
    ctx, orc = F.Context(log_n, q, [], 1, sampling="seeded"), O.Ctx(log_n, q, [], 1)
    rng = np.random.default_rng(19)
    pats = edge_patterns(q, ctx.n)
    half = pats[0].copy()  # last limb coefficient q_l / 2 and its neighbours
    last = q[-1]
    coef = np.array([last // 2, last // 2 + 1, last - 1, 0] * (ctx.n // 4), dtype=np.uint64)
    half[-1] = orc.ntt_fwd(coef, len(q) - 1)
    for a in [residues(rng, q, (2,), ctx.n), pats[1:3], np.stack([half, pats[3]])]:
        assert np.array_equal(ctx.rescale(ctx.upload(a)).numpy(), orc.rescale(a))
    ctx.close()


# (log_n, limbs, polys, ciphertexts, column kernel): batches on both sides of
# the line between three launches and four, and rings that have no such line.
BATCHES = [(14, 2, 2, 16, True), (17, 3, 1, 2, True), (13, 20, 2, 10, True), (13, 20, 2, 16, False), (14, 9, 2, 16, True),
           (14, 10, 2, 16, False), (14, 18, 2, 8, False), (14, 18, 2, 4, True),
           (15, 10, 2, 16, True), (16, 10, 2, 16, True)]


@pytest.mark.parametrize("log_n,nq,npoly,count,columns", BATCHES)
def test_rescale_batches(log_n, nq, npoly, count, columns):
    q = O.ntt_friendly_primes(log_n, 59, nq)
    ctx, orc = F.Context(log_n, q, [], 1, sampling="seeded"), O.Ctx(log_n, q, [], 1)
    rng = np.random.default_rng(29)
    xs = [residues(rng, q, (npoly,), ctx.n) for _ in range(2)]
    want = [orc.rescale(x) for x in xs]
    dev = [ctx.upload(xs[r % 2]) for r in range(count)]
    ctx.profile_begin()
    outs = ctx.rescale_many(dev)
    kernels = ctx.profile_end()
    for r, o in enumerate(outs):
        assert np.array_equal(o.numpy(), want[r % 2]), r
    assert ("k_rescale_mid" in kernels) is columns, kernels
    ctx.close()


# One ciphertext: 16 waves (more than 8 rounds of lines) at each column length
# that has that form, 8 at N=2^17, limb counts that do and do not fill a round.
SINGLES = [(13, 19), (13, 20), (14, 19), (14, 34), (15, 12), (15, 18), (16, 12), (17, 20),
           (17, 41)]


@pytest.mark.parametrize("log_n,nq", SINGLES)
def test_rescale_of_one_ciphertext(log_n, nq):
    q = O.ntt_friendly_primes(log_n, 59, nq)
    ctx, orc = F.Context(log_n, q, [], 1, sampling="seeded"), O.Ctx(log_n, q, [], 1)
    for npoly in (1, 2):
        x = residues(np.random.default_rng(31), q, (npoly,), ctx.n)
        assert np.array_equal(ctx.rescale(ctx.upload(x)).numpy(), orc.rescale(x)), npoly
    ctx.close()
