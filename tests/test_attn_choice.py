"""Which attention kernel runs (attn_plan.cpp), on both sides of the measured
lines; host arithmetic, no GPU."""
from attn_plan_util import plan


def test_short_kernel_range():
    """One sequence of up to 1024 rows on one kv head; with more heads while the
    rows of all heads or the walks over the keys stay few."""
    yes = [(1024, 3, 1), (1, 1, 1), (640, 4, 2), (640, 6, 2), (321, 4, 4), (384, 8, 4),
           (200, 8, 8), (256, 8, 8)]
    no = [(1025, 3, 1), (100, 4, 1), (641, 4, 2), (850, 4, 2), (400, 4, 4), (512, 8, 4),
          (257, 8, 8), (512, 8, 8)]
    for q, want in [(y, True) for y in yes] + [(n, False) for n in no]:
        assert (plan(*q).kind == "short") == want, q
    assert plan(300, 3, 1, segments=True).kind != "short"
    assert plan(300, 3, 1, hd=512).kind != "short"
