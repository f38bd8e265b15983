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
