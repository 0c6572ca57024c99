"""The planner's choices where they are close, by the launches that a call is mapped onto (no GPU; 256 compute units)."""
import pytest

from launch_routes import routes

BF16 = 0


@pytest.mark.parametrize("d", [104, 128])
def test_backward_of_41_to_64_sequences(d):
    """One launch of 64-column workgroups would take two rounds here (la_bwd, b*h = 48, n = 2048, d = 128: 97 us); dQ, then dK + dV
    paired, take 87.  Shared states only on longer walks; up to 40 sequences one launch is one round."""
    got = routes([(bh, n, d, d, BF16) for bh in (33, 40, 41, 48, 56, 64) for n in (256, 512, 1024, 1600, 2048, 3072, 3584, 5120, 8192)])
    for (bh, n, *_), r in got.items():
        if bh <= 40:
            assert ("once" in r["bwd"]) == (n <= 5120), (bh, n, r)
        elif n == 256:
            assert "once" in r["bwd"], (bh, n, r)  # (19.3 against 19.9)
        else:
            assert "once" not in r["bwd"] and ("shared" in r["bwd"]) == (n == 8192), (bh, n, r)
            assert n == 8192 or "sweep rev warm w0 x2 c1;" in r["bwd"], (bh, n, r)


@pytest.mark.parametrize("d, e", [(128, 96), (96, 128)])
def test_carried_dq_is_weighed_by_every_other_form(d, e):
    """d != e, states carried from the forward pass: la_bwd in one launch for dQ + dK, against a carried dQ, takes 155 / 138 us at
    b*h = 24, n = 6016, 282 / 270 at 48, 8192, but 155 / 163 at 48, 4096 and 238 / 265 at 64, 6016."""
    got = routes([(bh, n, d, e, BF16) for bh, n in ((24, 5120), (24, 6016), (32, 7168), (48, 8192), (48, 4096), (56, 6016), (64, 6016), (64, 12288))])
    for (bh, n, *_), r in got.items():
        if bh == 48 and n == 4096 or bh > 48:
            assert r["bwd"].startswith("dq+dk"), (bh, n, r)
        else:
            assert r["bwd"].startswith(("apply apply w1 x1", "trio")), (bh, n, r)


def test_saved_matrices_are_weighed_by_the_one_launch_form():
    """65 .. 80 sequences at d = 128: the forward pass leaves matrices, and from 40 blocks on the backward pass starts dQ from them
    rather than running everything in one launch (fwd + bwd of b*h = 72: n = 8192 528 / 549 us, n = 32768 2108 / 2246)."""
    got = routes([(bh, n, 128, 128, BF16) for bh in (65, 72, 80) for n in (2560, 4096, 32768)])
    for key, r in got.items():
        assert "saving" in r["fwd"] and "sweep resume" in r["bwd"], (key, r)


def test_long_walks_of_short_rows_read_no_more_than_they_must():
    """d = 64, 45 .. 64 sequences: one launch makes ten passes over a tensor, carried and shared states twelve: la_bwd of 64 sequences,
    n = 65536, 1065 / 1175 us.  With 41 sequences, or rows of 40, blocks still count: 465 / 436, 936 / 855."""
    got = routes([(bh, n, d, d, BF16) for bh, n, d in ((48, 8192, 64), (48, 49152, 64), (64, 24576, 64), (64, 65536, 64), (52, 24576, 64), (41, 32768, 64), (64, 65536, 40))])
    for (bh, n, d, *_), r in got.items():
        assert ("once" in r["bwd"]) == (d == 64 and bh > 41), (bh, n, d, r)


def test_one_launch_for_three_sweeps_of_different_rows():
    """d = 128, e = 64: three sweeps in one launch where that measures faster than dQ + dK in one and dV scanned."""
    got = routes([(bh, n, 128, 64, BF16) for bh, n in ((8, 2048), (8, 4096), (16, 2048), (16, 4096), (24, 6016), (40, 16384))])
    assert all(r["bwd"].startswith("trio") for r in got.values()), got
    got = routes([(bh, n, 128, 64, BF16) for bh, n in ((1, 5120), (8, 5120), (8, 6016), (16, 6016), (24, 12288), (24, 16384))] +
                 [(2, 6509, 80, 64, BF16), (10, 8192, 96, 64, BF16), (18, 10240, 80, 64, BF16), (32, 4096, 128, 40, BF16)])
    assert all(r["bwd"].startswith("dq+dk") for r in got.values()), got
    got = routes([(8, 4096, 64, 128, BF16), (24, 12288, 64, 128, BF16), (48, 16384, 64, 128, BF16), (24, 8192, 104, 64, BF16), (32, 3072, 128, 40, BF16), (16, 8192, 40, 96, BF16), (8, 6016, 40, 96, BF16)])
    assert all(r["bwd"].startswith("trio") for r in got.values()), got
    got = routes([(2, 6016, 64, 128, BF16), (8, 6016, 64, 128, BF16), (10, 8192, 64, 128, BF16), (2, 6016, 40, 96, BF16)])
    assert all("trio" not in r["bwd"] and r["bwd"].count("scan") == 3 for r in got.values()), got


def test_what_is_kept_is_read():
    """The forward pass leaves states (up to 21 MB a layer, for as long as the graph lives) only where the backward pass starts its dQ
    sweep from them."""
    pairs = ((128, 128), (104, 104), (96, 96), (64, 64), (40, 40), (192, 192), (128, 96), (72, 128), (64, 40), (192, 160), (128, 64))
    lengths = (64, 512, 1024, 1600, 2048, 3072, 4096, 6016, 8192, 12288, 16384, 24576, 37888, 65536)
    shapes = [(bh, n, d, e, BF16) for d, e in pairs for bh in (1, 8, 16, 24, 32, 40, 48, 56, 64, 72, 80, 88, 96, 128, 160) for n in lengths]
    kept = 0
    for once in (0, 1, 2):
        for key, r in routes(shapes, once=once).items():
            assert bool(r["kept"]) == ("carried" in r["bwd"] or "resume" in r["bwd"]), (once, key, r)
            kept += bool(r["kept"])
    assert kept > 500


def test_shapes_that_the_gpu_tests_mean_a_launch_by():
    """What tests/test_gpu_bwd_trio.py and tests/test_gpu_carried_states.py take their shapes to run."""
    pairs = [(48, 130, 128, 96), (48, 700, 96, 128), (41, 513, 72, 128), (88, 200, 64, 40), (128, 65, 32, 64)]
    for key, r in routes([p + (BF16,) for p in pairs]).items():
        assert r["bwd"].startswith("dq+dk warm w0") and "sweep rev warm" in r["bwd"], (key, r)
    carried = {(16, 8192, 128, 128, 0): 8, (13, 9057, 128, 128, 0): 8, (64, 6400, 128, 128, 0): 2, (16, 16384, 64, 64, 0): 8, (64, 4096, 128, 128, 0): 0,
               (45, 6113, 72, 72, 0): 0, (24, 6400, 96, 120, 1): 0, (9, 9001, 48, 40, 1): 0}
    for key, r in routes(carried).items():
        assert "carried" in r["bwd"] and ("x2 c%d shared" % carried[key] in r["bwd"] if carried[key] else "shared" not in r["bwd"]), (key, r)
    for key, r in routes([(16, 8192, 128, 128, 0), (64, 6400, 128, 128, 0)], workspace=False).items():
        assert "carried" in r["bwd"] and "sweep rev warm" in r["bwd"], (key, r)
