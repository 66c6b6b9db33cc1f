"""RungeKutta.Perform on the host with change rates that are not the library's: an override in a subclass or on the
instance, one that reads the stepper's state, and an operator with evaluate_dev alone."""
import numpy as np
import pytest
import torch

from bosss_amd.timestepping import RK4, TVD3, RungeKutta


class Decay:
    """R(U) = U through the accumulating evaluate."""

    def evaluate_dev(self, U, R, alpha=1.0, beta=0.0):
        R.mul_(beta).add_(U, alpha=alpha)


class Halved(RungeKutta):
    def ComputeChangeRate(self, k, U):
        k.add_(U, alpha=0.5)


class ReadsState(RungeKutta):
    def ComputeChangeRate(self, k, U):
        k.add_(self.U, alpha=0.5)


def on_instance(op, U, scheme):
    rk = RungeKutta(op, U, scheme)
    rk.ComputeChangeRate = lambda k, U: k.add_(U, alpha=0.5)
    return rk


@pytest.mark.parametrize("scheme,order", [(TVD3, 3), (RK4, 4)])
@pytest.mark.parametrize("make,rate", [(RungeKutta, 1.0), (Halved, 0.5), (ReadsState, 0.5), (on_instance, 0.5)])
def test_change_rates_of_the_caller(make, rate, scheme, order):
    U = torch.tensor([1.0, -2.0], dtype=torch.float64)
    U0, dt = U.clone(), 0.1
    rk = make(Decay(), U, scheme)
    for _ in range(2):
        assert rk.Perform(dt) == dt
    # the stability polynomial of an order-p scheme with p stages: sum_k (-rate dt)^k / k!
    z, growth, term = -rate * dt, 1.0, 1.0
    for k in range(1, order + 1):
        term *= z / k
        growth += term
    assert rk.U is U and abs(rk.time - 2 * dt) < 1e-15
    assert np.abs(U.numpy() - growth ** 2 * U0.numpy()).max() < 1e-14
