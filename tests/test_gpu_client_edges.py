"""Encode, encrypt, decrypt and decode at the edges of their kernels' ranges."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

F = pytest.importorskip("fhemamba_amd")


@pytest.fixture(scope="module", params=[(5, 3, 30), (12, 1, 45), (14, 2, 59), (16, 33, 45),
                                        (17, 2, 58)])
def pair(request):
    log_n, depth, sb = request.param
    q, p = O.gen_moduli(log_n, depth, sb, 60 if sb > 40 else 40, 1)
    ctx, orc = F.Context(log_n, q, p, 1, sampling="seeded"), O.Ctx(log_n, q, p, 1)
    yield ctx, orc
    ctx.close()


def close(got, want):
    """Both sides take up to 33 Horner steps and 16 transform stages on the
    same coefficients, each rounding by 2^-53 of values no larger than the
    results' norm: 2^-46 of it at most, 2^-40 of the largest result."""
    assert np.abs(got - want).max() <= 2.0**-40 * np.abs(want).max()


@pytest.mark.parametrize("log_slots", [0, 1, 5, 11, 12, 13, 16])
def test_encode_and_decode_by_slot_count(pair, log_slots):
    """One slot (no transform), one block of the block kernel, and 1 to 5 of
    the register kernel's stages; real, complex and short rows, one at a time
    and batched, equal the oracle's coefficients; decode agrees with the oracle's
    at one limb and at all of them."""
    ctx, orc = pair
    slots = 1 << log_slots
    if 2 * slots > ctx.n:
        pytest.skip("more slots than the ring holds")
    rng = np.random.default_rng(log_slots)
    scale = 2.0 ** 28
    real = rng.uniform(-2, 2, (3, slots))
    rows = real + 1j * rng.uniform(-2, 2, (3, slots))
    short = real[:, : (slots + 1) // 2]
    for nq in {1, ctx.L}:
        for z in (real, rows, short):
            want = [orc.encode(r, slots, scale, nq) for r in z]
            for w, one, many in zip(want, [ctx.encode(r, slots, scale, nq) for r in z],
                                    ctx.encode_many(z, slots, scale, nq)):
                assert np.array_equal(one.numpy()[0], w)
                assert np.array_equal(many.numpy()[0], w)
        close(ctx.decode(ctx.upload(want[0][None]), slots, scale),
              orc.decode(want[0], slots, scale))


def test_decode_of_residues_over_the_whole_range(pair):
    """Digits of either sign and largest size in every limb: the coefficients
    +-(q_j - 1) / 2 of each limb, 0, 1 and random residues.  A wrong digit
    makes every later one wrong and so the value's leading bits."""
    ctx, orc = pair
    rng = np.random.default_rng(9)
    slots = ctx.n // 2
    mods = ctx.q[:17]  # products beyond leave the range of doubles
    pt = np.stack([rng.integers(0, int(q), ctx.n, dtype=np.uint64) for q in mods])
    for i, q in enumerate(mods):
        pt[i, :4] = [0, 1, int(q) // 2, int(q) // 2 + 1]
    pt = np.stack([orc.ntt_fwd(r, i) for i, r in enumerate(pt)])
    close(ctx.decode(ctx.upload(pt[None]), slots, 2.0**60), orc.decode(pt, slots, 2.0**60))


def test_encrypt_and_decrypt_with_wide_signed_coefficients(pair):
    """Samples drawn on the device equal the oracle's; decryption lifts signed
    coefficients of any size, the extremes of int64 included."""
    ctx, orc = pair
    s = orc.secret(3)
    pk = orc.public_key(s, 4)
    rng = np.random.default_rng(2)
    m = np.stack([rng.integers(0, int(q), ctx.n, dtype=np.uint64) for q in ctx.q])
    for nq in {1, ctx.L}:
        ct = ctx.encrypt(ctx.upload(pk), ctx.upload(m[None, :nq].copy()), 6)
        assert np.array_equal(ct.numpy(), orc.encrypt(pk, m[:nq].copy(), 6))
        wide = rng.integers(-2**63, 2**63, ctx.n, dtype=np.int64)
        wide[:4] = [-2**63, 2**63 - 1, -int(ctx.q[0]), 0]
        zero_one = np.stack([np.zeros((nq, ctx.n), np.uint64), np.ones((nq, ctx.n), np.uint64)])
        got = ctx.decrypt(ctx.upload(zero_one), wide)  # 0 + 1 * s: the lifted s itself
        for i, q in enumerate(ctx.q[:nq]):
            lifted = (wide.astype(object) % int(q)).astype(np.uint64)
            assert np.array_equal(got.numpy()[0, i], orc.ntt_fwd(lifted, i))
