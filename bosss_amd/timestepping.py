"""Explicit Runge-Kutta time stepping on the device-resident operator (host mirror of
BoSSS.Solution.TimeStepping.ExplicitEuler / RungeKutta).

Convention of the reference: the operator gives the change rate R(u) of du/dt + R(u) = 0.
`ComputeChangeRate(k, U)` accumulates k += R(U) (`ExplicitEuler.cs:223-229`, an
Evaluate(1, 1, k) of the evaluator); a stage sets y = y0 - dt sum_r a[s][r] k[r]
(`RungeKutta.cs:297-310`), the step ends with y0 - dt sum_s b[s] k[s] (`RungeKutta.cs:242-285`).
Every vector stays on the GPU; one residual launch per stage.
"""
from .operator import DifferentialOperator


class RungeKuttaScheme:
    """Butcher tableau (a strictly lower triangular, b, c), as RungeKuttaScheme.cs."""

    def __init__(self, a, b, c):
        self.a, self.b, self.c = a, b, c
        self.stages = len(b)


# ExplicitEuler; TVD3 of Gottlieb and Shu (Math. Comp. 67 (1998) 73-85), the reference's
# RungeKuttaScheme.TVD3; the classic fourth-order scheme.
EXPLICIT_EULER = RungeKuttaScheme([[0.0]], [1.0], [0.0])
TVD3 = RungeKuttaScheme([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.25, 0.25, 0.0]], [1.0 / 6.0, 1.0 / 6.0, 2.0 / 3.0], [0.0, 1.0, 0.5])
RK4 = RungeKuttaScheme([[0.0] * 4, [0.5, 0.0, 0.0, 0.0], [0.0, 0.5, 0.0, 0.0], [0.0, 0.0, 1.0, 0.0]],
                       [1.0 / 6.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 6.0], [0.0, 0.5, 0.5, 1.0])


class RungeKutta:
    """Explicit Runge-Kutta stepper over a DifferentialOperator's device evaluate.

    `U` is the current state, updated in place.  A change rate of the caller's own (`ComputeChangeRate`
    overridden in a subclass or set on the instance, or an operator with its own `evaluate_dev`) is
    called once per stage with a zeroed k to add to, and finds the stage state in `U` itself, as in the
    reference (`RungeKutta.cs:297-310` writes it to the mapping's fields)."""

    def __init__(self, op, U, scheme=TVD3):
        import torch
        self.op, self.scheme = op, scheme
        self.U = U
        self.time = 0.0
        self.k = [torch.empty_like(U) for _ in range(scheme.stages)]
        self.y0 = torch.empty_like(U)                # the start of the step, or (fused updates) the stage states

    def ComputeChangeRate(self, k, U):
        """k += R(U)  (ExplicitEuler.ComputeChangeRate)."""
        self.op.evaluate_dev(U, k, alpha=1.0, beta=1.0)

    def Perform(self, dt):
        """One time step of size dt; returns dt (RungeKutta.Perform)."""
        if self._fused():
            self._perform_fused(dt)
        else:
            self._perform(dt)
        self.time += dt
        return dt

    def _fused(self):
        """Whether the change rate is this class's over the library's residual, so that nothing but this step
        sees k and the stage states."""
        op = self.op
        return (getattr(self.ComputeChangeRate, "__func__", None) is RungeKutta.ComputeChangeRate and isinstance(op, DifferentialOperator)
                and getattr(op.evaluate_dev, "__func__", None) is DifferentialOperator.evaluate_dev)

    def _perform(self, dt):
        sch = self.scheme
        self.y0.copy_(self.U)
        for s in range(sch.stages):
            if s > 0:
                # PerformStage: U = y0 - dt sum_r a[s][r] k[r]
                self.U.copy_(self.y0)
                for r in range(s):
                    if sch.a[s][r] != 0.0:
                        self.U.add_(self.k[r], alpha=-dt * sch.a[s][r])
            self.k[s].zero_()
            self.ComputeChangeRate(self.k[s], self.U)
        self.U.copy_(self.y0)
        for s in range(sch.stages):
            if sch.b[s] != 0.0:
                self.U.add_(self.k[s], alpha=-dt * sch.b[s])

    def _perform_fused(self, dt):
        """The same step with one pass per update: the stage states beside U (no copies of it), k written instead
        of zeroed and added to."""
        sch = self.scheme
        for s in range(sch.stages):
            y = self._combine(sch.a[s][:s], dt, self.y0)
            self.op.evaluate_dev(y, self.k[s])
        self._combine(sch.b, dt, self.U)

    def _combine(self, a, dt, out):
        """out <- U - dt sum_r a[r] k[r] over the coefficients that are not zero; returns where the result is
        (U itself if there are none)."""
        used = [r for r in range(len(a)) if a[r] != 0.0]
        if not used:
            return self.U
        self.op.combine_dev(self.U, [-dt * a[r] for r in used], [self.k[r] for r in used], out)
        return out
