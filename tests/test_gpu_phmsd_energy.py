"""The particle-hole energy kernel at the edges of its work split, against the oracle, to the
1e-10 bar of test_gpu_phmsd: slices in one, exactly full and one-over LDS runs, a single
excitation, fewer and more electrons than the eight lanes that share a slice, ranks up to six, more
configurations of one rank than threads, thousands of configurations with a number of vectors that
is no multiple of the opposite-spin kernel's eight or sixteen, and a slice that leaves a CU to one
workgroup.
"""
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_phmsd import TOL, gpu, rel, rel_log, say, setup_case  # noqa: E402,F401


@pytest.mark.parametrize("kw,W", [
    (dict(N=12, nel=3, M=1, ndet=2, ncore=1, nactive=5, max_rank=1, seed=31), 3),
    (dict(N=16, nel=5, M=31, ndet=30, ncore=0, nactive=9, max_rank=4, seed=32), 5),
    (dict(N=16, nel=5, M=32, ndet=30, ncore=0, nactive=9, max_rank=4, seed=33), 4),
    (dict(N=20, nel=9, M=33, ndet=50, ncore=2, nactive=12, max_rank=5, seed=34), 3),
    (dict(N=30, nel=12, M=17, ndet=900, ncore=2, nactive=20, max_rank=2, seed=35), 2),
    (dict(N=16, nel=6, M=20, ndet=150, ncore=0, nactive=14, max_rank=6, seed=37), 2),
    (dict(N=24, nel=8, M=26, ndet=6000, ncore=0, nactive=20, max_rank=2, seed=38), 2),
    (dict(N=66, nel=36, M=5, ndet=12, ncore=30, nactive=34, max_rank=3, seed=36), 2),
])
def test_energy(gpu, kw, W):  # noqa: F811
    afq, ctx, torch = gpu
    say(f"case: PHMSD energy {kw} W={W}")
    P, ph, ham, trial, ot, t = setup_case(afq, ctx, **kw)
    say("  nconf", ph.nconf, "max rank", ph.max_rank(0), ph.max_rank(1))
    Pa, Pb = P.walkers(W, seed=7, noise=0.3)
    E, ov = afq.empty((W, 3), torch.complex128), afq.empty(W, torch.complex128)
    trial.Energy(afq.WalkerSet(Pa, Pb), E, ov)
    Er, ovr = ot.energy(t["hblk"], t["Lblk"], Pa, Pb)
    assert rel(afq.host(E), Er) < TOL and rel_log(afq.host(ov), ovr) < TOL
