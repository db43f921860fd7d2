"""M-sweeps over a caller's order of meioses, the ignorable ones (a founder's only
child: no other order samples them) among them, against the oracle: a trio, whose
meioses are all ignorable, and a family with both kinds.  Planned launches size a
step by the jobs of the order's own meioses."""
import numpy as np
import pytest

from family_cases import family_case
from oracle_lib import Oracle
from swiftlink_amd import native

pytestmark = pytest.mark.gpu

# two founder couples, their three and two children, a marriage between, two
# married-in founders with one child each
WIDE = dict(mother=[-1] * 6 + [0, 0, 0, 2, 2, 6, 6, 4, 8], father=[-1] * 6 + [1, 1, 1, 3, 3, 9, 9, 7, 5], founders=6)
TRIO = dict(mother=[-1, -1, 0], father=[-1, -1, 1], founders=2)


@pytest.mark.parametrize("mode,chains", ((native.SL_MSAMPLER_TWO_LAUNCH, 3), (native.SL_MSAMPLER_AUTO, 70),
                                         (native.SL_MSAMPLER_SPECULATIVE, 3)))
@pytest.mark.parametrize("family,order", ((TRIO, [0, 1]), (TRIO, [1, 1]), (WIDE, "ignorable"), (WIDE, "all")))
def test_given_order_equals_the_oracle(family, order, mode, chains):
    case, g0 = family_case(markers=65, missing=0.4, seed=11, **family)
    o = Oracle(case)
    nm = 2 * (case.N - case.F)
    if isinstance(order, str):
        order = [b for b in range(nm) if order == "all" or b not in set(o.meioses())]
        assert len(order) >= 2
    order = np.array(order, np.int32)
    # flips that genotype elimination does not decide, at some locus, among them
    assert (case.geno == 0).any() and (case.geno == 1).any()
    with native.Context(case, native.SL_FP64, msampler_mode=mode) as ctx:
        ctx.mcmc_init(np.repeat(g0[None], chains, axis=0))
        for sweep in range(3):
            ctx.msweep(51, sweep, order)
        out = ctx.mcmc_graphs()
        assert np.all(ctx.mcmc_status() == 0)
        near = ctx.mcmc_near_edge()
    for c in sorted({0, 1, chains // 2, chains - 1}):
        g = g0
        for sweep in range(3):
            g = o.msweep(g, order, 51, c, sweep)
        assert near[c] == 0
        assert np.array_equal(out[c], g), c
