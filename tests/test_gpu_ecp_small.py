"""Channeling patterns of up to 64 strong beams, one workgroup per direction (ctem_ecp_small.hip), at
every padded size and its neighbour above (the batched products), with thicknesses whose first step differs
from the increment. Both modes sum in double; the oracle's exact integral and its Pade depth sum therefore
agree with the float32 intensities to 1 ulp."""
import numpy as np
import pytest

from ecp_cases import fixture, native_setup, oracle_crystal, setup_params

pytestmark = pytest.mark.gpu


def _ulps(a, b):
    ia, ib = (np.asarray(v, np.float32).view(np.int32).astype(np.int64) for v in (a, b))
    return np.abs(ia - ib)


@pytest.mark.parametrize("mode", ["Blochwv", "ScatMat"])
@pytest.mark.parametrize("key,weak,sizes", [("s1", 2.0, {32}), ("s1", 30.0, {32}), ("s1", 60.0, {32, 64}), ("s1", 100.0, {64, 96}),
                                            ("s1", 130.0, {96, 128}), ("s2", 8.0, {32}), ("s2", 40.0, {64}), ("s2", 60.0, {64, 96})])
def test_small_sets(key, weak, sizes, mode, oracle_mod, monkeypatch):
    import ecp_cases
    from ctemsoft_amd import ebsd, ecp
    z = fixture()
    cut = (weak, 2.0 * weak, 0.05)
    monkeypatch.setattr(ecp_cases, "setup_params", lambda *a: dict(setup_params(*a), cutoffs=cut))
    st, _, geo = native_setup(z, key)
    cr = oracle_crystal(z, key)
    occ = [s["occ"] for s in setup_params(z, key)["xtal"]["sites"]]
    thick = (np.float32(1.5) + np.float32(2.5) * np.arange(4, dtype=np.float32)).astype(np.float32)
    ctx = ebsd.Context(0)
    try:
        ctx.upload_crystal(st)
        p = ecp.EcpPlan(ctx, geo["k"], geo["kn"], mode, 1.5, 2.5, 4, 0.5, geo["dynfn"], occ)
        ns, _ = p.select()
        p.run()
        sr = p.sr()
    finally:
        ctx.close()
    assert np.isfinite(sr).all()
    assert set(((ns + 31) // 32 * 32).tolist()) == sizes
    order = np.argsort(ns, kind="stable")
    pick = np.unique(np.concatenate([order[[0, 1, -2, -1]], order[::max(1, len(order) // 8)]]))
    print(f"{key} {weak} {mode}: {ns.min()}..{ns.max()} beams, {len(pick)} directions", flush=True)
    for ik in pick:
        want, *_ = oracle_mod.ecp_direction(cr, geo["k"][ik], geo["kn"][ik], geo["dynfn"], mode, thick, 0.5,
                                            exact=mode == "Blochwv")
        assert _ulps(sr[:, ik], want).max() <= 1, (ns[ik], sr[:, ik], want)


@pytest.mark.parametrize("mode", ["Blochwv", "ScatMat"])
@pytest.mark.parametrize("key,weak", [("s1", 30.0), ("s1", 100.0), ("s1", 300.0)])
def test_timing_counts_the_products(key, weak, mode, monkeypatch):
    """ctem_plan_timing after a channeling-pattern run, below and above 64 beams: a time, and flops between the
    fewest and the most products that the mode can take per direction."""
    import ecp_cases
    from ctemsoft_amd import ebsd, ecp
    z = fixture()
    cut = (weak, 2.0 * weak, 0.05)
    monkeypatch.setattr(ecp_cases, "setup_params", lambda *a: dict(setup_params(*a), cutoffs=cut))
    st, _, geo = native_setup(z, key)
    occ = [s["occ"] for s in setup_params(z, key)["xtal"]["sites"]]
    ctx = ebsd.Context(0)
    try:
        ctx.upload_crystal(st)
        p = ecp.EcpPlan(ctx, geo["k"], geo["kn"], mode, 1.5, 2.5, 4, 0.5, geo["dynfn"], occ)
        ns, _ = p.select()
        p.run()
        first = p.timing()
        p.run()
        t = p.timing()
    finally:
        ctx.close()
    print(f"{weak} {mode}: {ns.min()}..{ns.max()} beams: {t}", flush=True)
    n3 = 8.0 * (ns.astype(float) ** 3).sum()
    assert t["gemm_ms"] > 0 and t["gemm_launches"] > 0 and t["gemm_ms"] <= t["total_ms"]
    assert t["gemm_flops"] == first["gemm_flops"]
    few, most = (32, 32 + 6 * 51) if mode == "Blochwv" else (1, 14 + 4)
    if ns.max() > 64:
        most *= 8
    assert few * n3 <= t["gemm_flops"] <= most * n3
