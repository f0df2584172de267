"""A program that replaces a part of the predictor or of its network gets that
part called: the fused calls, which stand for all of them, step aside.  Only the
choice is made here, before any device call."""
import pytest

torch = pytest.importorskip("torch")

from hpsint_amd.predictor import MLP, N_IN, N_OUT, LearnedPredictor  # noqa: E402


class Operator:
    handle, n_nodes, n_dofs = None, 8, 32


class Called(Exception):
    pass


def raising(*args, **kwargs):
    raise Called


def network(cls=MLP):
    return cls(Operator(), device="cpu")


@pytest.mark.parametrize("name", ["forward", "loss_grad", "backward", "adam"])
@pytest.mark.parametrize("where", ["subclass", "instance", "class"])
def test_training_step_calls_replaced_parts(monkeypatch, name, where):
    cls = type("Mine", (MLP,), {name: raising}) if where == "subclass" else MLP
    mlp = network(cls)
    X, T = torch.zeros(4, N_IN, dtype=torch.bfloat16), torch.zeros(4, N_OUT)
    parts = {"forward": (None, None), "loss_grad": (0.0, None), "backward": (None, None),
             "adam": None}
    for other, result in parts.items():          # the rest without a device
        if other != name:
            monkeypatch.setattr(mlp, other, lambda *a, r=result: r)
    if where == "instance":
        monkeypatch.setattr(mlp, name, raising)
    if where == "class":
        monkeypatch.setattr(MLP, name, raising)
    with pytest.raises(Called):
        mlp.train_step(X, T, 4, 1e-3)


@pytest.mark.parametrize("part", ["features", "forward", "network"])
def test_prediction_calls_replaced_parts(part):
    class Network:                               # not an MLP, but a forward()
        W = [torch.zeros(1)]
        forward = raising

    if part == "network":
        pred = LearnedPredictor(Operator(), Network())
    elif part == "forward":
        pred = LearnedPredictor(Operator(), network(type("Mine", (MLP,), {"forward": raising})))
    else:
        pred = type("Mine", (LearnedPredictor,), {"features": raising})(Operator(), network())
    if part != "features":
        pred.features = lambda *a: (None, None)
    u = [torch.zeros(Operator.n_dofs, dtype=torch.float64) for _ in range(3)]
    with pytest.raises(Called):
        pred.predict(u[0], u[1], 1e-3, u[2])


def test_each_part_alone_takes_the_parts():
    """one replaced part is enough"""
    X, T = torch.zeros(4, N_IN, dtype=torch.bfloat16), torch.zeros(4, N_OUT)
    for name in ("forward", "loss_grad", "backward", "adam"):
        assert network(type("Mine", (MLP,), {name: raising}))._train_fused(X, T, 4, 1e-3) is None
    u = [torch.zeros(Operator.n_dofs, dtype=torch.float64) for _ in range(3)]
    for pred in (LearnedPredictor(Operator(), network(type("Mine", (MLP,), {"forward": raising}))),
                 type("Mine", (LearnedPredictor,), {"features": raising})(Operator(), network())):
        assert pred._infer_workspace(*u) is None
