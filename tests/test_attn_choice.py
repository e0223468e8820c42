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


def test_partitioned_choices():
    """The fitted costs' choices at shapes measured on every choice: many short
    sequences and few q heads on 64-query blocks, short full layers on 16-query
    blocks, long ones on 32 x 32 tiles, and as many partitions as measured best
    (within one)."""
    for t, nq, nkv, hd, w, rows, kind in [
            (128, 4, 2, 256, 512, 8192, "q64"), (64, 1, 1, 256, 0, 6400, "q64"),
            (64, 4, 2, 256, 512, 6400, "q64"), (200, 3, 1, 256, 0, 3072, "q16"),
            (512, 3, 1, 256, 0, 16384, "q64"), (426, 3, 1, 256, 0, 5440, "tile"),
            (512, 4, 1, 512, 0, 16384, "tile"), (1500, 4, 1, 512, 0, 4608, "tile"),
            (512, 4, 1, 256, 0, 16384, "tile"), (400, 4, 4, 256, 0, 4480, "tile"),
            (128, 4, 4, 256, 0, 8192, "tile")]:
        p = plan(t, nq, nkv, hd, w, rows=rows, segments=True)
        assert (p.kind, p.kparts) == (kind, 1), (t, nq, nkv, hd, rows, p)
    for t, nq, nkv, hd, w, kind, kparts in [
            (8192, 3, 1, 256, 0, "q64", 2), (8192, 4, 1, 512, 0, "tile", 1),
            (3500, 3, 1, 256, 0, "tile", 3), (1777, 4, 2, 256, 512, "tile", 4),
            (1300, 3, 1, 256, 0, "tile", 6), (1300, 1, 1, 256, 0, "q64", 8),
            (1000, 4, 1, 256, 0, "q16", 4), (333, 4, 1, 512, 0, "q16", 6)]:
        p = plan(t, nq, nkv, hd, w)
        assert p.kind == kind and abs(p.kparts - kparts) <= 1, (t, nq, nkv, hd, p)
