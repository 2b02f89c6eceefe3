"""HIP path against the CPU oracle, through the C ABI.

The plain form follows the oracle's operation order, so match lists
(positions and order), distances, paste-mask decisions and model
eigenvalues are compared bit for bit; aggregation weights to 1e-6 relative
(exp/log are evaluated in double on both sides and can differ by one float
ulp in rare double-rounding cases); stage outputs within max-abs 1e-3 and
PSNR 0.02 dB (the plain-form tolerance), and in practice far closer.
"""
import numpy as np
import pytest
import torch

import vnlbhip
import workloads
from vnlbhip import synth
from vnlbhip.params import BASIC, FINAL, StageParameters, parse_stage_parameters

pytestmark = pytest.mark.gpu

MAX_ABS = 1e-3
PSNR_TOL = 0.02


def _dev(a):
    a = np.ascontiguousarray(a, np.float32)
    if a.ndim == 3:
        a = a[:, None]
    return torch.from_numpy(a).to("cuda:0")


def _compare_frame(gpu, oracle_lib, stage, params, noisy, ref, anchor_frame):
    want = oracle_lib.frame_debug(stage, params, noisy, ref, anchor_frame)
    got = gpu.debug_frame(stage, params, _dev(noisy), _dev(ref) if ref is not None else None,
                          anchor_frame)
    assert got["cap"] == want["cap"]
    np.testing.assert_array_equal(got["anchor_x"], want["anchor_x"])
    np.testing.assert_array_equal(got["anchor_y"], want["anchor_y"])
    np.testing.assert_array_equal(got["counts"], want["counts"])
    for a, n in enumerate(want["counts"]):
        np.testing.assert_array_equal(got["positions"][a, :n], want["positions"][a, :n])
        np.testing.assert_array_equal(got["distances"][a, :n], want["distances"][a, :n])
    np.testing.assert_array_equal(got["active"], want["active"])
    np.testing.assert_array_equal(got["group_flags"], want["group_flags"])
    act = want["active"] == 1
    modelled = act & ((want["group_flags"] & 4) != 0)
    np.testing.assert_array_equal(got["eigenvalues"][modelled], want["eigenvalues"][modelled])
    for a in np.nonzero(act)[0]:
        n = want["counts"][a]
        np.testing.assert_allclose(got["weights"][a, :n], want["weights"][a, :n], rtol=1e-6, atol=0)
    return want


def _check_output(got, want, clean=None):
    got = got.cpu().numpy() if torch.is_tensor(got) else got
    diff = np.abs(got - want)
    assert diff.max() <= MAX_ABS, f"max abs {diff.max()}"
    if clean is not None:
        assert abs(synth.psnr(got, clean) - synth.psnr(want, clean)) <= PSNR_TOL
    return float(diff.max())


@pytest.mark.parametrize("name", list(workloads.WORKLOADS))
def test_match_paste_model_bitwise(gpu, oracle_lib, name):
    noisy, clean, bp, fp = workloads.make(name)
    print(f"[parity] {name} {noisy.shape}", flush=True)
    frames = noisy.shape[0]
    for af in sorted({0, 1, frames - bp.patch_time}):
        _compare_frame(gpu, oracle_lib, BASIC, bp, noisy, None, af)
    basic, _ = oracle_lib.stage(BASIC, bp, noisy, flags=oracle_lib.ACCUM_DOUBLE, threads=4)
    for af in sorted({0, 2, frames - fp.patch_time}):
        _compare_frame(gpu, oracle_lib, FINAL, fp, noisy, basic, af)


@pytest.mark.parametrize("patch_size,group_size", [
    (8, 2), (8, 3), (8, 4), (8, 5), (8, 8), (8, 9), (8, 12), (8, 13), (8, 16), (8, 17), (8, 31), (8, 32), (8, 33),
    (8, 63), (8, 64), (8, 65), (8, 100), (8, 112), (9, 90), (11, 122), (3, 40), (5, 60)])
def test_eigen_solver_sizes(gpu, oracle_lib, patch_size, group_size):
    """Eigen problems at the edges of the solvers' sizes (4, 8, 12, 16, 32, 64
    and 128 rows), dual (8x8x2 patches) and covariance (121, 81, 25 and 9 samples per
    patch) ones: eigenvalues bit for bit, weights from the eigenvectors."""
    noisy, _ = synth.make_clip(40, 36, 4, 1, sigma8=15, seed=90 + group_size, motion="subpixel")
    args = dict(sigma=15, block_size=patch_size, block_step=6, group_size=group_size, bm_range=6, radius=1, tau=0,
                patch_time=2 if patch_size == 8 else 1, rank=min(group_size, 20, patch_size * patch_size))
    bp = parse_stage_parameters(BASIC, args)
    print(f"[parity] {patch_size}x{patch_size} patches, {group_size} neighbours", flush=True)
    want = _compare_frame(gpu, oracle_lib, BASIC, bp, noisy, None, 1)
    assert ((want["group_flags"] & 4) != 0).any()


@pytest.mark.parametrize("name", list(workloads.WORKLOADS))
def test_stage_outputs(gpu, oracle_lib, name):
    noisy, clean, bp, fp = workloads.make(name)
    print(f"[stage] {name} {noisy.shape}", flush=True)
    want_basic, groups = oracle_lib.stage(BASIC, bp, noisy, flags=oracle_lib.ACCUM_DOUBLE, threads=4)
    got_basic = gpu.stage(BASIC, bp, _dev(noisy))
    assert gpu.stats()["groups"] == groups
    _check_output(got_basic, want_basic, clean)
    # Final on the same guide clip, then the chained GPU form.
    want_final, _ = oracle_lib.stage(FINAL, fp, noisy, want_basic, flags=oracle_lib.ACCUM_DOUBLE, threads=4)
    got_final = gpu.stage(FINAL, fp, _dev(noisy), _dev(want_basic))
    _check_output(got_final, want_final, clean)
    chained = gpu.stage(FINAL, fp, _dev(noisy), got_basic)
    _check_output(chained, want_final, clean)
    # The reference's float-order accumulation stays within the tolerance too.
    ref_order_basic, _ = oracle_lib.stage(BASIC, bp, noisy, flags=0, threads=4)
    _check_output(got_basic, ref_order_basic, clean)


@pytest.mark.parametrize("case", range(6))
def test_pariasm_fixture_cases(gpu, oracle_lib, case):
    name, noisy, basic_ref, final_ref, bp, fp, tol = workloads.pariasm_cases()[case]
    print(f"[pariasm] {name}", flush=True)
    want_basic, _ = oracle_lib.stage(BASIC, bp, noisy, flags=oracle_lib.ACCUM_DOUBLE)
    got_basic = gpu.stage(BASIC, bp, _dev(noisy))
    _check_output(got_basic, want_basic)
    got_final = gpu.stage(FINAL, fp, _dev(noisy), got_basic)
    want_final, _ = oracle_lib.stage(FINAL, fp, noisy, want_basic, flags=oracle_lib.ACCUM_DOUBLE)
    _check_output(got_final, want_final)
    for got, ref in ((got_basic, basic_ref), (got_final, final_ref)):
        diff = np.abs(got.cpu().numpy()[:, 0] - ref)
        assert diff.max() <= tol["max_abs"] and diff.mean() <= tol["mean_abs"]
        assert np.sqrt((diff ** 2).mean()) <= tol["rmse"]
    _compare_frame(gpu, oracle_lib, BASIC, bp, noisy, None, 1)


def test_integer_valued_clip_is_exact(gpu, oracle_lib):
    """Samples on a 1/16 lattice make every distance exact in any order;
    ties are everywhere, so this pins the (distance, scan position) order."""
    noisy = workloads.integer_clip()
    p = StageParameters(sigma=10 / 255, patch_size=4, patch_time=1, search_window=7, search_bwd=1,
                        search_fwd=1, similar=8, rank=4, proc_step=2, tau=0.05)
    _compare_frame(gpu, oracle_lib, BASIC, p, noisy, None, 1)
    want, _ = oracle_lib.stage(BASIC, p, noisy, flags=oracle_lib.ACCUM_DOUBLE)
    got = gpu.stage(BASIC, p, _dev(noisy)).cpu().numpy()
    assert np.abs(got - want).max() <= 1e-6


def _nan_clip():
    rng = np.random.default_rng(17)
    noisy = rng.random((4, 1, 48, 64), dtype=np.float32)
    noisy[:, :, :, :24] = np.nan
    return noisy


def test_nan_region_anchors_are_skipped(gpu, oracle_lib):
    """Anchors whose every candidate distance is NaN have no matches: they
    form no group and clear nothing (the oracle skips them), and their
    pixels fall back to the (NaN) source."""
    noisy = _nan_clip()
    p = StageParameters(sigma=20 / 255, patch_size=4, patch_time=1, search_window=7, search_bwd=1,
                        search_fwd=1, similar=8, rank=4, proc_step=2)
    print("[nan] debug frame", flush=True)
    want_dbg = _compare_frame(gpu, oracle_lib, BASIC, p, noisy, None, 1)
    assert (want_dbg["counts"] == 0).any() and (want_dbg["counts"] > 0).any()
    print("[nan] stage", flush=True)
    want, groups = oracle_lib.stage(BASIC, p, noisy, flags=oracle_lib.ACCUM_DOUBLE)
    got = gpu.stage(BASIC, p, _dev(noisy)).cpu().numpy()
    assert gpu.stats()["groups"] == groups
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    finite = ~np.isnan(want)
    assert np.abs(got[finite] - want[finite]).max() <= MAX_ABS


@pytest.mark.parametrize("group_size,patch_time", [(3, 2), (12, 2), (24, 2), (40, 2), (70, 1)])
def test_infinite_sample_in_the_models(gpu, oracle_lib, group_size, patch_time):
    """An infinite chroma sample, which Basic does not match on, leaves models
    with infinite and NaN diagonals: every eigenpair still has a place, and
    the output is the oracle's (its tolerance above, the sample itself
    aside) at each of the solver's sizes."""
    noisy, _ = synth.make_clip(48, 40, 4, 3, sigma8=15, seed=31, motion="subpixel")
    noisy = noisy.copy()
    noisy[1, 1, 20, 24] = np.inf
    p = parse_stage_parameters(BASIC, dict(sigma=15, block_size=8, block_step=4, group_size=group_size, bm_range=5,
                                           patch_time=patch_time, radius=1, rank=min(group_size, 8), tau=0, chroma=1))
    print(f"[inf] {group_size} neighbours", flush=True)
    want, _ = oracle_lib.stage(BASIC, p, noisy, flags=oracle_lib.ACCUM_DOUBLE)
    got = gpu.stage(BASIC, p, _dev(noisy)).cpu().numpy().reshape(want.shape)
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(want))
    finite = np.isfinite(want)
    assert np.abs(got[finite] - want[finite]).max() <= MAX_ABS


def test_constant_clip(gpu):
    noisy = np.full((3, 1, 24, 20), 0.25, np.float32)
    p = StageParameters(sigma=0.1, patch_size=2, patch_time=1, search_window=3, search_bwd=1,
                        search_fwd=1, similar=4, rank=4, beta=2.0, tau=1000.0, proc_step=2)
    out = gpu.stage(BASIC, p, _dev(noisy)).cpu().numpy()
    np.testing.assert_allclose(out, 0.25, atol=1e-5)
    out = gpu.stage(FINAL, p, _dev(noisy), _dev(noisy)).cpu().numpy()
    np.testing.assert_allclose(out, 0.25, atol=1e-5)


def test_single_patch_groups_and_fallback(gpu):
    noisy, _ = synth.make_clip(40, 32, 3, 1, sigma8=10, seed=2)
    p = StageParameters(sigma=10 / 255, patch_size=4, patch_time=1, search_window=5, similar=1,
                        rank=0, proc_step=9)
    out = gpu.stage(BASIC, p, _dev(noisy)).cpu().numpy()
    np.testing.assert_allclose(out, noisy, atol=1e-6)


def test_host_buffer_entry_point(gpu, oracle_lib):
    noisy, clean, bp, fp = workloads.make("gray_p8_step8")
    noisy = noisy[:, :, :64, :80]
    got = gpu.stage(BASIC, bp, noisy)  # numpy in -> vnlbhip_stage_host
    want, _ = oracle_lib.stage(BASIC, bp, noisy, flags=oracle_lib.ACCUM_DOUBLE)
    _check_output(got, want)


def test_invalid_parameters_raise(gpu):
    import vnlbhip

    noisy = _dev(np.zeros((4, 1, 32, 32), np.float32))
    p = StageParameters(sigma=0.1, rank=32, similar=16, patch_time=1)
    with pytest.raises(vnlbhip.VNLBError, match="group_size must cover the effective VNLB rank"):
        gpu.stage(BASIC, p, noisy)


@pytest.mark.parametrize("channels,extra", [
    # Groups of one round of samples, the tile over the basis (YUV rank 16).
    (3, dict(group_size=16, rank=16)),
    # Groups that widen past one round there (no tile), and past one round of a tile of its own.
    (3, dict(group_size=16, rank=16, tau=200000)),
    (3, dict(group_size=10, rank=2, tau=200000)),
    (1, dict(group_size=8, rank=8, tau=200000)),
    (3, dict(group_size=9, rank=4, tau=200000, chroma=0)),
    # More samples than a round by the group size itself.
    (1, dict(group_size=40, rank=12)),
    # Windows too wide for a tile, single-sample groups, one to four patch frames.
    (3, dict(group_size=16, rank=4, bm_range=18)),
    (1, dict(group_size=1, rank=1)),
    (1, dict(group_size=16, rank=6, patch_time=1)),
    (1, dict(group_size=16, rank=6, patch_time=3)),
    (1, dict(group_size=16, rank=6, patch_time=4)),
    # Unit aggregation window, rank 0.
    (3, dict(group_size=16, rank=0, weight_gamma=0.0))])
def test_aggregation_paths(gpu, oracle_lib, channels, extra):
    """Every way a group's samples reach the accumulators, on a width that is
    no multiple of a memory line.  Both sides add the same float products in
    double; the weights agree to 1e-6 relative (see above) and samples stay
    below 2 in magnitude, so the weighted means differ by at most 2 * 2e-6 and
    a float rounding: 5e-6."""
    noisy, _ = synth.make_clip(61, 45, 5, channels, sigma8=5, seed=123, motion="subpixel")
    args = dict(dict(sigma=15, block_size=8, block_step=5, bm_range=7, patch_time=2, radius=1, tau=0), **extra)
    bp, fp = parse_stage_parameters(BASIC, args), parse_stage_parameters(FINAL, args)
    print(f"[parity] aggregation {channels} {extra}", flush=True)
    want_basic, _ = oracle_lib.stage(BASIC, bp, noisy, flags=oracle_lib.ACCUM_DOUBLE, threads=4)
    want_final, _ = oracle_lib.stage(FINAL, fp, noisy, want_basic, flags=oracle_lib.ACCUM_DOUBLE, threads=4)
    basic = gpu.stage(BASIC, bp, _dev(noisy))
    if args["tau"] > 0:
        stats = gpu.stats()
        assert stats["retained"] > 1.5 * args["group_size"] * stats["groups"]
    final = gpu.stage(FINAL, fp, _dev(noisy), _dev(want_basic))
    for got, want in ((basic, want_basic), (final, want_final)):
        assert np.abs(got.cpu().numpy().reshape(want.shape) - want).max() <= 5e-6


@pytest.mark.parametrize("form", ["plain", "fast"])
@pytest.mark.parametrize("width,height,frames,extra", [
    # 81 k anchors: past the joined lists of small batches.
    (138, 131, 5, dict(block_size=8, block_step=1, group_size=8, rank=8, bm_range=2)),
    # 22 k anchors of 112-row models: past their bytes.
    (76, 72, 6, dict(block_size=8, block_step=1, group_size=112, rank=8, bm_range=5, patch_time=2))])
def test_batches_of_separate_group_lists(oracle_lib, form, width, height, frames, extra):
    """Batches whose parts keep their group lists and model launches: the
    oracle's groups; outputs within the plain form's tolerance, 0.05 dB in
    the fast one."""
    noisy, clean = synth.make_clip(width, height, frames, 1, sigma8=15, seed=77, motion="subpixel")
    p = parse_stage_parameters(BASIC, dict(dict(sigma=15, radius=1, tau=0, patch_time=1), **extra))
    print(f"[parity] separate lists, {form}, {width}x{height}x{frames}", flush=True)
    ctx = vnlbhip.Context(0)
    try:
        ctx.set_form(form)
        got = ctx.stage(BASIC, p, _dev(noisy)).cpu().numpy()
        stats = ctx.stats()
    finally:
        ctx.close()
    want, groups = oracle_lib.stage(BASIC, p, noisy, flags=oracle_lib.ACCUM_DOUBLE, threads=4)
    assert stats["parts"] > 1
    if form == "plain":
        assert stats["groups"] == groups
        _check_output(got.reshape(want.shape), want, clean)
    else:
        assert abs(synth.psnr(got.reshape(want.shape), clean) - synth.psnr(want, clean)) <= 0.05
