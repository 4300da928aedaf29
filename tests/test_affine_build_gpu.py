"""GPU: the affine reset's chunk maps at the edges of the build's tiles, rows and slots: chunks that
are no multiple of the 32-step tile, neuron counts around the 16 of a workgroup, maps of more than
16 pieces (a lane's second slot) that shrink below it again, and overflows at every capacity,
against the oracle's maps bit for bit."""
import numpy as np
import pytest
import torch

from oracle import affine_oracle as A
from tests._inputs import gpu, host, normal, uniform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,K,N", [(1, 32, 15), (33, 32, 16), (100, 17, 17), (130, 32, 33), (64, 16, 1),
                                   (200, 31, 20)])
@pytest.mark.parametrize("gamma,delta,beta,mu,sd", [(1.0, -1.0, 0.99, -0.1, 0.6), (0.9, -0.8, 0.97, 0.1, 0.7),
                                                    (0.0, -0.2, 0.95, 0.15, 0.4)])
def test_build_matches_oracle(dev, C, K, N, gamma, delta, beta, mu, sd):
    from lifscan import triton_affine as AF
    T = 5 * C
    I, u0 = normal(T, N, mu, sd, C), uniform(N, -1.0, 1.0, 7)
    keep, sto, st = {}, {}, {}
    print(f"affine build C={C} K={K} N={N} gamma={gamma}", flush=True)
    Uo, So = A.scan_forward(I, beta, 1.0, gamma, delta, u0, C=C, K=K, stats=sto, keep=keep)
    U, S = AF.aff_scan_forward(gpu(I, dev), beta, 1.0, gamma, delta, gpu(u0, dev), C=C, K=K, stats=st)
    run = AF.last_aff_run()
    assert np.array_equal(host(run.view("LO")), keep["Lo"])
    assert np.array_equal(host(run.view("HI")), keep["Hi"])
    assert np.array_equal(host(run.view("NP", torch.int32)), keep["n"])
    assert np.array_equal(host(run.view("OVF", torch.int32)), keep["ovf"])
    P = host(run.view("PIECES"))
    for f, name in enumerate(("xl", "xr", "a", "c")):
        assert np.array_equal(P[..., f], keep[name]), name
    assert np.array_equal(host(run.view("STARTS")), keep["starts"])
    assert np.array_equal(host(U), Uo) and np.array_equal(host(S), So)
    assert st["overflow_frac"] == pytest.approx(sto["overflow_frac"], abs=1e-12)
    assert st["mean_pieces"] == pytest.approx(sto["mean_pieces"], abs=1e-9)


# more than 768 workgroups of 16 neurons: a 16-lane row a neuron (above, 32 lanes)
@pytest.mark.parametrize("C,K,N,M", [(33, 32, 33, 260), (20, 17, 17, 400), (64, 16, 1, 780), (40, 31, 20, 400)])
@pytest.mark.parametrize("gamma,delta,beta,mu,sd", [(1.0, -1.0, 0.99, -0.1, 0.6), (0.9, -0.8, 0.97, 0.1, 0.7),
                                                    (0.0, -0.2, 0.95, 0.15, 0.4)])
def test_build_of_many_chunks_matches_oracle(dev, C, K, N, M, gamma, delta, beta, mu, sd):
    from lifscan import triton_affine as AF
    I, u0 = normal(M * C, N, mu, sd, C), uniform(N, -1.0, 1.0, 7)
    keep, sto, st = {}, {}, {}
    print(f"affine build M={M} C={C} K={K} N={N} gamma={gamma}", flush=True)
    Uo, So = A.scan_forward(I, beta, 1.0, gamma, delta, u0, C=C, K=K, stats=sto, keep=keep)
    U, S = AF.aff_scan_forward(gpu(I, dev), beta, 1.0, gamma, delta, gpu(u0, dev), C=C, K=K, stats=st)
    run = AF.last_aff_run()
    assert np.array_equal(host(run.view("NP", torch.int32)), keep["n"])
    assert np.array_equal(host(run.view("OVF", torch.int32)), keep["ovf"])
    P = host(run.view("PIECES"))
    for f, name in enumerate(("xl", "xr", "a", "c")):
        assert np.array_equal(P[..., f], keep[name]), name
    assert np.array_equal(host(U), Uo) and np.array_equal(host(S), So)
    assert st["mean_pieces"] == pytest.approx(sto["mean_pieces"], abs=1e-9)
