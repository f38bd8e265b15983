"""Key switches whose ModUp digits are used once (their last forward pass runs
inside ModDown's) against those of shared digits, which keep the separate
pass, and against the oracle."""
import numpy as np
import pytest

import oracle as O
from gpu_helpers import edge_patterns, residues

pytestmark = pytest.mark.gpu
F = pytest.importorskip("fhemamba_amd")


# (log_n, Q limbs, P limbs, dnum): 1 to 4 digits, a ragged last digit, 5 and 8
# digits (past the rule), every block-pass length.
@pytest.mark.parametrize("log_n,L,K,dnum", [(13, 4, 4, 1), (13, 7, 4, 2), (14, 8, 3, 3),
                                            (15, 7, 2, 4), (15, 9, 2, 5), (13, 8, 1, 8),
                                            (16, 7, 2, 4), (16, 5, 2, 3), (17, 5, 3, 2)])
def test_single_use_digits(log_n, L, K, dnum):
    q = O.ntt_friendly_primes(log_n, 58, L)
    p = O.ntt_friendly_primes(log_n, 59, K, skip=q)
    ctx, orc = F.Context(log_n, q, p, dnum, sampling="seeded"), O.Ctx(log_n, q, p, dnum)
    rng = np.random.default_rng(log_n * 100 + L)
    keys = [residues(rng, list(q) + list(p), (ctx.dnum, 2), ctx.n) for _ in range(2)]
    dkeys = [ctx.load_key(k) for k in keys]
    gal = [5, 2 * ctx.n - 1, 1]
    use = [dkeys[0], dkeys[1], dkeys[0]]
    for nq in range(1, L + 1):
        cts = [residues(rng, q[:nq], (2,), ctx.n) for _ in range(3)]
        pats = edge_patterns(q[:nq], ctx.n)
        cts[2] = np.stack([pats[1], pats[2]])
        dev = [ctx.upload(c) for c in cts]
        want = [ctx.rotate_hoisted(d, ctx.rotation_precompute(d), [k], [g])[0].numpy()
                for d, k, g in zip(dev, use, gal)]
        for w, got in zip(want, ctx.rotate_many(dev, use, gal)):
            assert np.array_equal(got.numpy(), w), nq
        for w, d, k, g in zip(want, dev, use, gal):
            assert np.array_equal(ctx.rotate(d, k, g, out=d).numpy(), w), nq
        if nq in (1, L):
            assert np.array_equal(want[0], orc.rotate(cts[0], keys[0], gal[0]))
            ct3 = residues(rng, q[:nq], (3,), ctx.n)
            assert np.array_equal(ctx.relinearize(ctx.upload(ct3), dkeys[1]).numpy(),
                                  orc.relinearize(ct3, keys[1]))
    ctx.close()


@pytest.mark.parametrize("log_n,L,K,dnum,count,inside", [
    (13, 3, 1, 3, 1, False), (13, 4, 1, 4, 2, False), (14, 7, 2, 4, 1, False),
    (15, 4, 1, 4, 1, False), (13, 2, 1, 2, 1, True), (13, 4, 1, 4, 32, True),
    (16, 3, 1, 3, 1, True)])
def test_small_switches_keep_the_digits_pass(log_n, L, K, dnum, count, inside):
    """Three or four digits of 5 MiB or less in all are finished by a pass of
    their own, whose chain is shorter; the others inside ModDown."""
    q = O.ntt_friendly_primes(log_n, 58, L)
    p = O.ntt_friendly_primes(log_n, 59, K, skip=q)
    ctx, orc = F.Context(log_n, q, p, dnum, sampling="seeded"), O.Ctx(log_n, q, p, dnum)
    rng = np.random.default_rng(5)
    key = residues(rng, list(q) + list(p), (ctx.dnum, 2), ctx.n)
    dkey = ctx.load_key(key)
    ct = residues(rng, q, (2,), ctx.n)
    cts = [ctx.upload(ct) for _ in range(count)]
    ctx.profile_begin()
    outs = ctx.rotate_many(cts, [dkey] * count, [5] * count)
    kernels = ctx.profile_end()
    want = orc.rotate(ct, key, 5)
    for o in outs:
        assert np.array_equal(o.numpy(), want)
    assert ("ntt_fwd_blocks_modup" in kernels) is not inside, kernels
    ctx.close()
