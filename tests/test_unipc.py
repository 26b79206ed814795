"""UniPC flow-matching sampler: the oracle (oracle/unipc_oracle.py) against what the mathematics fixes, and
the torch scheduler (longlive_amd/utils/unipc.py) against the oracle.  CPU only."""
import math

import numpy as np
import pytest
import torch
from scipy.integrate import quad

import unipc_oracle as uo
from longlive_amd.utils import unipc
from longlive_amd.utils.unipc import FlowUniPCMultistepScheduler, convert_flow_pred_to_x0


def test_schedule_closed_form():
    sig, ts = uo.schedule(4, 1.0)
    assert np.allclose(sig, [0.999, 0.74925, 0.4995, 0.24975, 0.0], atol=1e-7) and list(ts) == [999, 749, 499, 249]
    assert list(uo.schedule(6, 1.0)[1]) == [999, 832, 666, 499, 333, 166]  # 666: sigma_max is float32(0.999) > 0.999
    sig5, ts5 = uo.schedule(4, 5.0)
    assert np.allclose(sig5[:-1], [5 * s / (1 + 4 * s) for s in sig[:-1]]) and sig5[-1] == 0.0
    sch = FlowUniPCMultistepScheduler(num_train_timesteps=1000, shift=1)
    sch.set_timesteps(4, shift=5.0)
    assert np.allclose(sch.sigmas.numpy(), sig5, atol=1e-7) and sch.timesteps.tolist() == list(ts5)


def test_phi_functions_and_weights():
    for z in (-3.0, -0.7, -1e-3, 0.4, 2.0):
        assert math.isclose(uo.phi(1, z), math.expm1(z) / z, rel_tol=1e-12)
        # phi_(k+1)(z) = integral_0^1 e^{(1 - t) z} t^k / k! dt
        for k in (1, 2, 3):
            ref = quad(lambda t: math.exp((1 - t) * z) * t ** k / math.factorial(k), 0, 1)[0]
            assert math.isclose(uo.phi(k + 1, z), ref, rel_tol=1e-9)


def _exact_solution(x_s, sigma_s, sigma_t, m_of_lambda):
    """x_t = (sigma_t / sigma_s) x_s + sigma_t * integral exp(lambda) m(lambda) d lambda (data prediction)."""
    ls, lt = uo.lam(sigma_s), uo.lam(sigma_t)
    integral = quad(lambda l: math.exp(l) * m_of_lambda(l), ls, lt, epsabs=1e-13, epsrel=1e-13)[0]
    return sigma_t / sigma_s * x_s + sigma_t * integral


def test_first_order_is_the_exponential_integrator():
    x_s, m = 0.37, -1.2
    for sigma_s, sigma_t in ((0.999, 0.75), (0.5, 0.25), (0.9, 0.1)):
        got = uo.uni_p(x_s, [m], [sigma_s], sigma_t, 1)
        h = uo.lam(sigma_t) - uo.lam(sigma_s)
        assert math.isclose(got, sigma_t / sigma_s * x_s - (1 - sigma_t) * math.expm1(-h) * m, rel_tol=1e-13)
        assert math.isclose(got, _exact_solution(x_s, sigma_s, sigma_t, lambda l: m), rel_tol=1e-10)
    assert uo.uni_p(x_s, [m], [0.25], 0.0, 1) == m  # the last step returns the x0 prediction


@pytest.mark.parametrize("coeffs", [(0.8, -0.5, 0.0), (0.3, 1.1, -0.7)])
def test_second_order_corrector_is_exact_for_quadratics_in_lambda(coeffs):
    """UniC-2 uses the previous node, the step's start and the predicted point: three nodes, exact up to
    degree 2.  A wrong R, b, phi recurrence or node position breaks this."""
    c0, c1, c2 = coeffs
    sigma_prev, sigma_s, sigma_t = 0.8, 0.6, 0.35
    ls = uo.lam(sigma_s)
    m = lambda l: c0 + c1 * (l - ls) + c2 * (l - ls) ** 2
    x_s = 0.21
    got = uo.uni_c(x_s, [m(uo.lam(sigma_prev)), m(ls)], [sigma_prev, sigma_s], sigma_t, m(uo.lam(sigma_t)), 2)
    assert math.isclose(got, _exact_solution(x_s, sigma_s, sigma_t, m), rel_tol=1e-9)
    # the order-1 corrector (fixed weight 1/2) is exact for constants only
    got1 = uo.uni_c(x_s, [m(ls)], [sigma_s], sigma_t, m(uo.lam(sigma_t)), 1)
    assert (abs(got1 - _exact_solution(x_s, sigma_s, sigma_t, m)) < 1e-9) == (c1 == 0 and c2 == 0)


def test_constant_x0_prediction_is_reproduced_by_every_step():
    rng = np.random.default_rng(0)
    x0, noise = rng.standard_normal(8), rng.standard_normal(8)
    sig, _ = uo.schedule(4, 5.0)
    x = (1 - sig[0]) * x0 + sig[0] * noise
    traj = uo.sample(lambda x, s, t: (x - x0) / s, x, 4, 5.0)  # flow = noise - x0 along the straight line
    for i, xi in enumerate(traj):
        assert np.allclose(xi, (1 - sig[i + 1]) * x0 + sig[i + 1] * noise, atol=1e-12)
    assert np.allclose(traj[-1], x0, atol=1e-12)


@pytest.mark.parametrize("steps,shift", [(4, 5.0), (6, 1.0), (3, 3.0), (1, 5.0)])
def test_torch_scheduler_follows_the_oracle(steps, shift):
    rng = np.random.default_rng(steps)
    A = rng.standard_normal((12, 12)) * 0.3
    flow_np = lambda x, s, t: np.tanh(x @ A) + 0.1 * s - 0.001 * (t % 7)
    x0 = rng.standard_normal((2, 12))
    want = uo.sample(flow_np, x0.copy(), steps, shift)
    sch = FlowUniPCMultistepScheduler(num_train_timesteps=1000, shift=1)
    sch.set_timesteps(steps, shift=shift)
    x = torch.from_numpy(x0).float()
    for i, t in enumerate(sch.timesteps):
        flow = torch.from_numpy(flow_np(x.double().numpy(), float(sch.sigmas[i]), int(t))).float()
        x = sch.step(flow, t, x, return_dict=False)[0]
        assert np.allclose(x.numpy(), want[i], atol=2e-5, rtol=2e-5), i
    assert sch.step_index == steps
    with pytest.raises(IndexError):
        fresh = FlowUniPCMultistepScheduler()
        fresh.set_timesteps(4)
        fresh.step(x, torch.tensor(123), x)


def test_scheduler_keeps_the_sample_dtype_and_rejects_unbuilt_modes():
    sch = FlowUniPCMultistepScheduler()
    sch.set_timesteps(4, shift=5.0)
    x = torch.randn(1, 3, 4, 4, generator=torch.Generator().manual_seed(0)).bfloat16()
    for t in sch.timesteps:
        x = sch.step(torch.randn_like(x), t, x).prev_sample
        assert x.dtype == torch.bfloat16 and torch.isfinite(x).all()
    with pytest.raises(NotImplementedError):
        FlowUniPCMultistepScheduler(solver_type="rk4")
    with pytest.raises(NotImplementedError):
        FlowUniPCMultistepScheduler(predict_x0=False)
    with pytest.raises(ValueError):
        FlowUniPCMultistepScheduler().step(x, 0, x)


def test_flow_to_x0_conversion():
    xt = torch.tensor([[1.0, -2.0]], dtype=torch.bfloat16)
    flow = torch.tensor([[0.5, 0.25]], dtype=torch.bfloat16)
    out = convert_flow_pred_to_x0(flow, xt, 0.75)
    assert out.dtype == torch.bfloat16 and torch.equal(out, torch.tensor([[0.625, -2.1875]]).bfloat16())


def _sigma_of(lmbda):
    return 1.0 / (1.0 + math.exp(lmbda))


@pytest.mark.parametrize("which", ["predictor_order_2", "corrector_order_1"])
def test_the_fixed_weight_one_half_is_what_makes_the_step_second_order(which):
    """The order-2 predictor and the order-1 corrector do not solve for their single weight; the reference
    writes 1/2 (wan_5b/utils/fm_solvers_unipc.py:461-463, 603-604).  What determines that number: with a
    difference of two x0 predictions as the only correction term, the local error of a step of size h in lambda
    falls like h^3 for the weight 1/2 and only like h^2 for any other.  Measured on an x0 prediction that is
    linear in lambda: halving h divides the error by ~8 for the oracle's step, and by ~4 when the correction
    term is rescaled to a weight of 0.45 or 0.55."""
    c0, c1, x_s, lam_s = 0.3, 0.9, 0.21, 0.4
    m = lambda l: c0 + c1 * (l - lam_s)

    def errors(h):
        s_prev, s_s, s_t = _sigma_of(lam_s - h), _sigma_of(lam_s), _sigma_of(lam_s + h)
        exact = _exact_solution(x_s, s_s, s_t, m)
        first_order = uo.uni_p(x_s, [m(lam_s)], [s_s], s_t, 1)
        if which == "predictor_order_2":
            step = uo.uni_p(x_s, [m(lam_s - h), m(lam_s)], [s_prev, s_s], s_t, 2)
        else:
            step = uo.uni_c(x_s, [m(lam_s)], [s_s], s_t, m(lam_s + h), 1)
        correction = step - first_order  # the term that carries the weight 1/2
        return {w: first_order + correction * (w / 0.5) - exact for w in (0.5, 0.45, 0.55)}

    coarse, fine = errors(0.2), errors(0.1)
    assert 6.5 < coarse[0.5] / fine[0.5] < 9.5, coarse[0.5] / fine[0.5]
    for w in (0.45, 0.55):
        assert 2.8 < coarse[w] / fine[w] < 5.5, (w, coarse[w] / fine[w])
        assert abs(fine[w]) > 5 * abs(fine[0.5])


@pytest.mark.gpu
@pytest.mark.parametrize("shape,steps,order,solver", [((48, 3, 8, 32), 4, 2, "bh2"), ((1,), 5, 2, "bh1"), ((257,), 3, 1, "bh2"),
                                                      ((16, 33), 6, 2, "bh2"), ((5, 8), 1, 2, "bh2")])
def test_one_launch_step_has_the_bits_of_the_tensor_expressions(gpu, monkeypatch, shape, steps, order, solver):
    """The step as one launch against the same scheduler's tensor expressions on the GPU, whole trajectories with all
    history; lengths with and without whole 16-byte pieces, and an input that is not 16-byte aligned."""
    def run(fused):
        sch = FlowUniPCMultistepScheduler(num_train_timesteps=1000, shift=1, solver_order=order, solver_type=solver)
        sch.set_timesteps(steps, device=gpu, shift=5.0)
        calls, original = [], FlowUniPCMultistepScheduler._fused_step
        with monkeypatch.context() as m:
            m.setattr(FlowUniPCMultistepScheduler, "_fused_step",
                      lambda self, *a: calls.append(original(self, *a) if fused else None) or calls[-1])
            g = torch.Generator().manual_seed(5)
            pad = torch.randn(math.prod(shape) + 1, generator=g).bfloat16().to(gpu)
            x, trace = pad[1:].view(shape), []
            x[..., 0] = 0.0
            for t in sch.timesteps.tolist():
                flow = torch.randn(shape, generator=g).bfloat16().to(gpu) * 3
                x = sch.step(flow, t, x, return_dict=False)[0]
                trace += [x, sch.model_outputs[-1], sch.last_sample]
        assert all((c is not None) == fused for c in calls) and len(calls) == steps
        return trace

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    sch = FlowUniPCMultistepScheduler(shift=1)   # gradients and other types keep torch's own operations
    sch.set_timesteps(2, device=gpu)
    flow = torch.ones(4, device=gpu, dtype=torch.bfloat16, requires_grad=True)
    assert sch.step(flow, sch.timesteps[0], torch.ones_like(flow), return_dict=False)[0].requires_grad


@pytest.mark.gpu
@pytest.mark.parametrize("method", ["convert_model_output", "_predict", "_correct"])
def test_step_calls_the_methods_put_in_place_of_its_own(gpu, method):
    """A scheduler whose pieces of a step are a subclass's runs them instead of the one launch."""
    calls = []

    def replacement(self, *args):
        calls.append(method)
        return getattr(super(Mine, self), method)(*args) + 1

    Mine = type("Mine", (FlowUniPCMultistepScheduler,), {method: replacement})
    outs = []
    for cls in (FlowUniPCMultistepScheduler, Mine):
        sch = cls(shift=1)
        sch.set_timesteps(3, device=gpu, shift=5.0)
        x = torch.zeros(16, device=gpu, dtype=torch.bfloat16)
        for t in sch.timesteps:
            x = sch.step(torch.ones_like(x), t, x, return_dict=False)[0]
        outs.append(x)
    assert len(calls) == (2 if method == "_correct" else 3) and not torch.equal(*outs)


def test_scalars_of_a_step_do_not_depend_on_the_default_device():
    """They are kept per schedule, so the first call must not leave another device's arithmetic behind."""
    args = (0.6, 0.8, (0.9,), 2, "bh2", True)
    unipc._step_scalars.cache_clear()
    want = unipc._step_scalars(*args)
    unipc._step_scalars.cache_clear()
    with torch.device("meta"):
        assert unipc._step_scalars(*args) == want
