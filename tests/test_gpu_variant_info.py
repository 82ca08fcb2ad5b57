"""What se_variant_info says of the kernels that step_blocked takes."""
import pytest

import sandengine_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,side,least", [("four_materials", 256, 9), ("twelve_materials", 2048, 9)])
def test_sliced_runs_are_named(name, side, least):
    ctx = S.Context(0)
    rs = S.RuleSet(ctx, S.bundled_ruleset(name))
    w = S.World(ctx, rs, side, side)
    lds = w.variant_info(2, 0)[0]
    assert w.variant_info(4, least - 1) == (0, 0, 0)
    takes, kernel, deep = w.variant_info(4, least)
    assert takes == 1 and 0 <= kernel < 4 and 1 <= deep <= least
    assert w.variant_info(4, 1000)[2] <= 32
    w.set_variant(3, lds)  # an LDS variant by name
    assert w.variant_info(4, 1000) == (0, 0, 0)
    last = lds
    while True:
        try:
            last, named = last + 1, w.variant_info(3, last + 1)[1]
        except S.SandengineError:
            break
    assert named == 0  # the last one names the sliced kernels, for any run
    w.set_variant(3, last)
    assert w.variant_info(4, 1)[0] == 1
    w.set_variant(3, -1)
    with pytest.raises(S.SandengineError):
        w.variant_info(4, 0)
    w.set_render(True)  # every step is a launch of its own
    assert w.variant_info(4, 1000) == (0, 0, 0)
    w.close()
