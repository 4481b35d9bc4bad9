"""bench.py's own figures and switches, without a GPU."""
import bench


def test_issued_matrix_products():
    """One v_mfma_scale_f32_16x16x128 per 16 weight rows, K step of 128 and
    activation term: the columns of all products together are the matrices'
    elements times their terms."""
    elements = {"glu": 2 * bench.INTER * bench.HIDDEN, "down": bench.HIDDEN * bench.INTER}
    want = elements["glu"] * bench.X_TERMS + elements["down"] * bench.H_TERMS
    assert bench._mfma_issued_per_expert() * 16 * 128 == want


def test_cpu_leg_needs_its_library(monkeypatch):
    """Without the reference's CPU library the line comes out with null baselines
    instead of ending at the first of them."""
    import oracle
    for there, asked in ((True, True), (True, False), (False, True), (False, False)):
        monkeypatch.setattr(oracle, "ref_available", lambda: there)
        assert bench.cpu_leg(asked) == (there and asked)


def test_spine_launch_time_of_either_kernel():
    gemv, mfma = {"total_ms": 0.24, "launches": 24}, {"total_ms": 0.36, "launches": 24}
    assert abs(bench.spine_launch_us({"spine_gemv": gemv}) - 10.0) < 1e-9
    assert abs(bench.spine_launch_us({"spine_mfma": mfma, "rms_norm": gemv}) - 15.0) < 1e-9
    assert abs(bench.spine_launch_us({"spine_gemv": gemv, "spine_mfma": mfma}) - 12.5) < 1e-9
