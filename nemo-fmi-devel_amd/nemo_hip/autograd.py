"""torch.autograd wrapper of the tracer step and its hand-written adjoint.

The tracer step is the one the adjoint entry points of the C-ABI transpose
(include/nemo_hip.h, "Tangent linear and adjoint of the tracer step"): for
one tracer in FP64, tra_adv_fct (orders kn) with the limiter factors of
nonosc (TRA/traadv_fct.F90:404-426), tra_ldf_lap, tra_zdf_imp and the
leapfrog tra_nxt, the velocities and diffusivities fixed.  Forward computes
the factors of the state and applies them (nemo_hip_tra_adv_fct_coef_tl), which
is the nonlinear step bit for bit; backward applies the adjoint entry points
with those factors frozen (the transpose of the step linearised with the
limiter held).  Nothing here computes: every operation is a library call on
resident device tensors, in order on the library stream.

run() steps a window and, with `every`, keeps only the state at every
`every`-th step: the backward pass recomputes each segment from its
checkpoint (torch.utils.checkpoint), so memory holds one segment's states.
"""
import torch
import torch.utils.checkpoint as tcp

from . import NEMO_HIP_PTR_DEVICE


class TracerModel:
    """The fixed fields of the tracer step: transports (zun, zvn, zwn of
    tra_adv), lateral diffusivities, vertical diffusivity, time step, FCT
    orders and the time-step index (kt > nit000: a leapfrog step)."""

    def __init__(self, h, zun, zvn, zwn, ahtu, ahtv, avt, p2dt, kn=(4, 4), kt=5):
        if h.mode != NEMO_HIP_PTR_DEVICE:
            raise ValueError("the autograd wrapper works on resident fields (device-pointer mode)")
        self.h, self.zun, self.zvn, self.zwn = h, zun, zvn, zwn
        self.ahtu, self.ahtv, self.avt = ahtu, ahtv, avt
        self.p2dt, self.kn, self.kt = float(p2dt), tuple(kn), kt
        self.n3 = zun.numel()
        self.stream = torch.cuda.ExternalStream(h.stream())

    def _z(self, n=1):
        return torch.zeros(n * self.n3, dtype=torch.float64, device="cuda")

    def factors(self, tb, tn):
        c = [self._z() for _ in range(3)]
        self.h.tra_adv_fct_coef(self.p2dt, self.zun, self.zvn, self.zwn, tb, tn, *c, kn=self.kn)
        return c

    def step(self, c, tb, tn):
        """one step with the limiter factors c: (tb, tn) -> (tb', tn')"""
        ta = self._z()
        self.h.tra_adv_fct_tl(self.p2dt, self.zun, self.zvn, self.zwn, tb, tn, *c, ta, kn=self.kn)
        return self._diffuse_and_swap(tb, tn, ta)

    def factors_and_step(self, tb, tn):
        """factors(tb, tn) and step with them, the fluxes evaluated once"""
        c, ta = [self._z() for _ in range(3)], self._z()
        self.h.tra_adv_fct_coef_tl(self.p2dt, self.zun, self.zvn, self.zwn, tb, tn, *c, ta, kn=self.kn)
        return c, self._diffuse_and_swap(tb, tn, ta)

    def _diffuse_and_swap(self, tb, tn, ta):
        h = self.h
        h.tra_ldf_lap(self.kt, 1, "TRA", self.ahtu, self.ahtv, tb, ta, 1, 1)
        h.tra_zdf_imp(self.kt, 1, "TRA", self.p2dt, tb, ta, 1, self.avt, self.avt)
        nb, nn = torch.empty_like(ta), torch.empty_like(ta)
        nb.copy_(tb)
        nn.copy_(tn)
        h.tra_nxt_one(self.kt, nb, nn, ta)
        return nb, nn

    def step_ad(self, c, lb, ln):
        """the adjoint of step with the factors c frozen: (lb', ln') -> (lb, ln)"""
        h = self.h
        lb, ln = lb.contiguous().clone(), ln.contiguous().clone()
        la = torch.empty_like(lb)   # tra_nxt_ad sets all of it
        h.tra_nxt_ad(lb, ln, la)
        h.tra_zdf_imp_ad(self.p2dt, self.avt, la, lb)
        h.tra_ldf_lap_ad(self.ahtu, self.ahtv, la, lb)
        h.tra_adv_fct_ad(self.zun, self.zvn, self.zwn, *c, la, lb, ln, kn=self.kn)
        return lb, ln


class TracerStep(torch.autograd.Function):
    """(tb, tn) -> (tb', tn') of one tracer step; backward: the adjoint with
    the forward step's limiter factors frozen."""

    @staticmethod
    def forward(ctx, tb, tn, model):
        cur = torch.cuda.current_stream()
        model.stream.wait_stream(cur)          # the inputs are ready
        with torch.cuda.stream(model.stream):
            c, (nb, nn) = model.factors_and_step(tb, tn)
        cur.wait_stream(model.stream)          # the outputs are ready
        for t in (nb, nn):
            t.record_stream(cur)
        ctx.model, ctx.c = model, c
        return nb, nn

    @staticmethod
    def backward(ctx, gb, gn):
        model = ctx.model
        cur = torch.cuda.current_stream()
        model.stream.wait_stream(cur)
        with torch.cuda.stream(model.stream):
            lb, ln = model.step_ad(ctx.c, model._z() if gb is None else gb, model._z() if gn is None else gn)
        cur.wait_stream(model.stream)
        for t in (lb, ln):
            t.record_stream(cur)
        return lb, ln, None


def _segment(model, steps):
    def f(tb, tn):
        for _ in range(steps):
            tb, tn = TracerStep.apply(tb, tn, model)
        return tb, tn
    return f


def run(model, tb, tn, steps, every=None):
    """`steps` tracer steps from (tb, tn), differentiable; with `every`, the
    states between checkpoints are recomputed in the backward pass"""
    if not every:
        return _segment(model, steps)(tb, tn)
    done = 0
    while done < steps:
        k = min(every, steps - done)
        tb, tn = tcp.checkpoint(_segment(model, k), tb, tn, use_reentrant=False)
        done += k
    return tb, tn
