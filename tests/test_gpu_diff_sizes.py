"""The differentiable form at the sizes it is used at (a picture of 1024 x 1024 with 256 paths,
512 x 512 with 128 paths of analytic coverage) against its float64 restatement: the picture
within the rounding of its sums, and most entries of the gradients as near, which the kinks
of the model (a clamped colour, a pixel's side of an edge) do not hide."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,batch,sigma", [("planes_1024", 1, 4.0), ("planes_1024", 1, 11.5),
                                              ("analytic_16x512", 2, 2.5)])
def test_picture_and_gradients_against_float64(ctx, name, batch, sigma):
    from perf import cases
    case = dict(next(c for c in cases.listed() if c["name"] == name), sigma=sigma)
    if "batch" in case:
        case["batch"] = batch
    got, want = cases.run(cases.prepare(case, 31)), cases.exact(case, 31)
    # a pixel passes `paths` composites of about 4 roundings, each at most 2^-24 of a value in
    # [0, 1]; independent, they add as their root
    rounding = 4.0 * case["paths"] ** 0.5 * 2.0 ** -24
    bound = rounding
    if case["kind"] == "analytic":
        # and the outlines' points are up to max(w, h) pixels with a float's 24 bits: through
        # the flattening's about 8 roundings an edge moves, and with it the coverage of a
        # pixel that it crosses
        bound += 8.0 * max(case["w"], case["h"]) * 2.0 ** -24
    image = got["image"].double() - want["image"]
    err = (image.norm() / want["image"].norm()).item()
    assert err < bound
    for key in [k for k in want if k != "image"]:
        d = (got[key].double() - want[key]).flatten()
        rms = want[key].norm().item() / d.numel() ** 0.5
        assert d.abs().median().item() < rounding * rms, key
