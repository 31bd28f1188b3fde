"""The sliced 16-latent fp32 form at the sizes where its loop can go wrong:
key ranges of 9 to 14 tiles of 16 (its tile loop runs in threes behind a first
tile, with a remainder of zero to two), whole and partial last tiles, a last
split of one key, of a tile and one key, and latents around a block of 16."""

import numpy as np
import pytest

from conftest import fp32_gate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nl", [1, 16, 17])
@pytest.mark.parametrize("ni", [129, 143, 144, 145, 160, 161, 175, 176, 192, 193, 208, 224])
def test_tile_counts(cw, oracle, nl, ni):
    q, k, v = oracle.make_inputs(2, nl, ni, 768, seed=100 + ni)
    out, _, _ = cw.benchmark_plan_events(q, k, v, 2, nl, ni, 768, 16, 1, warmup=1, iters=0)
    fp32_gate(out, oracle.attention_f64(q, k, v))


@pytest.mark.parametrize("nl, splits, keys, rest",
                         [(16, 145, 144, rest) for rest in (1, 15, 16, 17, 48)]
                         + [(17, 128, 129, rest) for rest in (2, 15, 16, 17, 48)])
def test_short_last_split(cw, oracle, nl, splits, keys, rest):
    """Splits of 9 tiles, the last of which has ``rest`` keys only (its window
    clamped or shifted, its look-ahead past its end), with a whole latent block
    and a block of one latent; the partials against the oracle's.  The counts
    are ones that the planner gives 16 latents per workgroup."""
    ni = (splits - 1) * keys + rest
    assert -(-ni // splits) == keys
    cu, _ = cw.device_info()
    if cu == 256:
        assert cw.lib.xattn_f32_split_latents(1, nl, ni, splits, cu) == 16
    q, k, v = oracle.make_inputs(1, nl, ni, 768, seed=rest)
    out, (po, pm, pl) = cw.splitk_partials(q, k, v, 1, nl, ni, 768, splits)
    fp32_gate(out, oracle.attention_f64(q, k, v))
    s = (q[0].astype(np.float64) @ k[0, -rest:].astype(np.float64).T) / np.sqrt(768.0)
    m = s.max(axis=1)
    e = np.exp(s - m[:, None])
    assert np.allclose(pm[0, :, -1], m, rtol=1e-5, atol=1e-5)
    assert np.allclose(pl[0, :, -1], e.sum(axis=1), rtol=1e-4)
    assert np.allclose(po[0, :, -1], e @ v[0, -rest:].astype(np.float64), rtol=1e-3, atol=1e-4)


def test_scores_that_outgrow_the_first_tile(cw, oracle):
    """Keys growing along the range force the passes to restart in every
    remainder of the loop.  Scores reach 200, so their own rounding shows: a
    score's error is taken as one rounding at the size of the sum of its
    products' magnitudes, 2^-24 sum |q k| / sqrt(D), and an output moves by at
    most twice that times the largest |v|."""
    for ni in (150, 165, 180):
        q, k, v = oracle.make_inputs(1, 16, ni, 768, seed=7)
        k = (k * np.linspace(1.0, 60.0, ni, dtype=np.float32)[None, :, None]).astype(np.float32)
        out, _, _ = cw.benchmark_plan_events(q, k, v, 1, 16, ni, 768, 16, 1, warmup=1, iters=0)
        score_err = 2.0 ** -24 * np.max(np.abs(q[0]) @ np.abs(k[0]).T) / np.sqrt(768.0)
        fp32_gate(out, oracle.attention_f64(q, k, v),
                  atol=float(2.0 * score_err * np.max(np.abs(v))))


@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("key", [5, 77, 149, 299])
def test_nan_stays_where_the_reference_puts_it(cw, oracle, key, splits):
    """As the fp32 tests' case of that name, over ranges that take this form
    (19 tiles of 16, or two splits of 10 and 9): a NaN in one batch element's K
    makes that element's whole output NaN, in its V only one column; every
    other value matches.  The key sits in the first tile, in the loop, in the
    last tile of a split and in a partial last tile, whose window repeats keys
    of the tile before."""
    b, nl, ni = 3, 17, 300
    for where in ("K", "V"):
        q, k, v = oracle.make_inputs(b, nl, ni, 768, seed=79)
        (k if where == "K" else v)[1, key, 5] = np.nan
        ref = oracle.attention_f64(q, k, v)
        nan = np.isnan(ref)
        assert nan[1].any() and not nan[[0, 2]].any()
        out, _, _ = cw.benchmark_plan_events(q, k, v, b, nl, ni, 768, 16, splits, warmup=1,
                                             iters=0)
        assert np.array_equal(np.isnan(out), nan), f"NaN in {where}: NaN pattern"
        fp32_gate(np.where(nan, 0.0, out), np.where(nan, 0.0, ref))
