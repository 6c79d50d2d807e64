"""The engine's step kernels and the pair kernels at the sizes where their splits can go
wrong: edges of tiles, spans and wavefronts, remainders, both ends of their ranges."""
import numpy as np
import pytest

from molecular_simulation_code_amd import system as S

pytestmark = pytest.mark.gpu


def _host():
    from molecular_simulation_code_amd import _lib
    if _lib.device_count() < 1:
        pytest.skip("no HIP device")
    from molecular_simulation_code_amd import host
    return host


@pytest.mark.parametrize("ng,nw", [(1, 1063), (2, 1060), (1, 1117), (63, 1000), (64, 1000), (65, 1000)])
def test_constraints_hold_at_span_and_wavefront_edges(ng, nw):
    """One atom short of, at and past a whole number of 160-atom spans, and 63 / 64 / 65
    clusters of each iterated kind.  Rigid waters are solved in closed form (1e-8 A); the other
    clusters to the solver's 1e-4 tolerance on lambda, a bond-length change of
    (1/m1 + 1/m2) r 1e-4 < 1.3e-4 A (below 3e-4 with the coupling of three constraints)."""
    host = _host()
    s = S.make_system(ng, nw, seed=100 + ng)
    e = host.Engine([host.ReplicaSpec(s, temp=300.0, gamma_ps=1.0, seed=3)])
    try:
        e.init()
        e.minimize(60)
        e.run(4)
        x, _ = e.state()[0]
    finally:
        e.close()
    L = float(s.box)
    a, b, d = S.constraint_pairs(s)
    r = x[a] - x[b]
    r -= L * np.round(r / L)
    err = np.abs(np.sqrt((r * r).sum(1)) - d)
    water = s.moltype[a] == 2
    print(f"[constraints] {s.np} atoms: water {err[water].max():.2e}, glycine {err[~water].max():.2e} A",
          flush=True)
    assert err[water].max() < 1e-8
    assert err[~water].max() < 3e-4
