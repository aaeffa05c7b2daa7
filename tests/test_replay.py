"""Which passes are replayed from a recorded plan and which go through the layer code: host logic, no GPU needed."""
from types import SimpleNamespace

import pytest
import torch

from bamboo_amd import hip, replay
from bamboo_amd.engine import PipelineEngine
from bamboo_amd.layers import FinalLayerNorm, StageContext

ROWS, COLS = 6, 8


class FakePlan:
    """Stands in for the native plan: counts replays and remembers what they were given."""

    launches = []

    class _Recording:
        made = None

        def __enter__(self):
            return FakePlan() if self.made is None else self.made

        def __exit__(self, *exc):
            return False

    @classmethod
    def record(cls):
        return cls._Recording()

    def dropout(self, keys):
        pass

    def operands(self, ranges):
        self.n = len(ranges)

    def launch(self, step, stream, tensors=()):
        FakePlan.launches.append([t.data_ptr() for t in tensors])


class FakeGraph(FakePlan):
    @classmethod
    def capture(cls, stream):
        recording = cls._Recording()
        recording.made = cls()
        return recording

    def launch(self, stream):
        FakePlan.launches.append(None)


class Layer(FinalLayerNorm):
    """A layer whose passes check their operands like the wrappers of the kernels do, and count."""

    launches_only = True
    feature_dim = out_features = COLS

    def forward(self, x, st, ctx):
        ctx.calls.append(("forward", self.eps))
        hip._like("forward", x, out=st["out"])
        st["x0"] = x
        return st["out"]

    def backward(self, d_out, d_x, st, ctx):
        ctx.calls.append(("backward", self.eps))
        hip._like("backward", d_out, out=st["out"], d_x=d_x, x0=st["x0"])
        return d_x


@pytest.fixture
def stage(monkeypatch):
    """An engine of one stage over CPU tensors: one layer, one micro-batch, passes called by hand."""
    from bamboo_amd.module import PipelineModule
    monkeypatch.setattr(hip, "Plan", FakePlan)
    monkeypatch.setattr(hip, "Graph", FakeGraph)
    FakePlan.launches = []
    module = object.__new__(PipelineModule)
    flat, arena = torch.zeros(64), torch.zeros(ROWS * COLS)
    layer = Layer(COLS)
    module.__dict__.update(loss_fn=None, base_seed=3, micro_offset=0, activation_checkpoint_interval=0, dtype=torch.float32,
                           func_buckets={1: [layer]}, _stash={1: [[{"out": arena.view(ROWS, COLS)}]]}, _stash_arena={1: arena}, stage_seq={1: [ROWS, ROWS]},
                           stage_params={1: SimpleNamespace(compute=flat, grad=flat)})
    ctx = StageContext(1, ROWS, torch.float32, "cpu")
    ctx.calls = []
    engine = object.__new__(PipelineEngine)
    lens, graphs = [None], {}
    engine.__dict__.update(
        module=module, ctx=ctx, rc_ctx=ctx, use_graphs=False, replay=True, _graphs=graphs, _replay=replay.Replay(module, graphs), global_steps=0, num_stages=3, stage_id=1, stage_ids=[1],
        r_stage_ids=[], rc_stream=None, rc_issue="reference", eager_recovery=False, _deferred={}, grad_layer={}, main_stream=None, device="cpu",
        queue=SimpleNamespace(key_len=lambda k: lens[0]), pipe_buffers={"input_1": [None], "output_1": [None], "input_grad_1": [None]},
        _input_grad_store={1: [torch.zeros(ROWS, COLS)]})

    def forward(x, key_len=None):
        lens[0] = key_len
        engine.pipe_buffers["input_1"][0], engine.pipe_buffers["output_1"][0] = x, None
        engine._exec_forward_pass(0, 1)
        return engine.pipe_buffers["output_1"][0]

    def backward(grad, key_len=None):
        lens[0] = key_len
        engine.grad_layer[1] = grad
        engine._exec_backward_pass(0, 1)
        return engine.pipe_buffers["input_grad_1"][0]
    return SimpleNamespace(engine=engine, module=module, layer=layer, ctx=ctx, forward=forward, backward=backward,
                           replayed=lambda: len(FakePlan.launches), issued=lambda: len(ctx.calls))


def test_other_buffers_of_the_same_form_are_replayed(stage):
    a, b = torch.randn(ROWS, COLS), torch.randn(ROWS, COLS)
    out = stage.forward(a)
    assert (stage.issued(), stage.replayed()) == (1, 0)
    assert stage.forward(b) is out and (stage.issued(), stage.replayed()) == (1, 1)
    assert FakePlan.launches[-1] == [b.data_ptr()]
    assert stage.module.kept_input(1, 0) is b and stage.module.micro_offset == 2
    d_x = stage.backward(a)
    for g in (b, a):
        assert stage.backward(g) is d_x
        assert FakePlan.launches[-1] == [g.data_ptr(), d_x.data_ptr(), b.data_ptr()]
    assert stage.issued() == 2 and all(len(v) == 1 for v in stage.engine._replay.plans.values())


# operands in a place that a recorded pass knows, which the layer code refuses
WRONG = {"rows": lambda t: t[: ROWS - 1], "columns": lambda t: t.view(-1)[: ROWS * (COLS - 4)].view(ROWS, COLS - 4),
         "type": lambda t: t.view(torch.int32).view(torch.float16)[:, :COLS], "strides": lambda t: t.view(COLS, ROWS).t()}


@pytest.mark.parametrize("graphs", [False, True], ids=["plans", "graphs"])
@pytest.mark.parametrize("wrong", list(WRONG))
def test_an_operand_of_another_form_in_a_known_place_is_refused(stage, wrong, graphs):
    x, g = torch.randn(ROWS, COLS), torch.randn(ROWS, COLS)
    stage.engine.use_graphs = graphs
    for _ in range(3):
        stage.forward(x)
        stage.backward(g)
    replays = stage.replayed()
    assert replays == 4
    bad_x, bad_g = WRONG[wrong](x), WRONG[wrong](g)
    assert bad_x.data_ptr() == x.data_ptr() and bad_g.data_ptr() == g.data_ptr()
    with pytest.raises(hip.HipKernelError):
        stage.backward(bad_g)
    with pytest.raises(hip.HipKernelError):
        stage.forward(bad_x)
    assert stage.replayed() == replays


def test_key_lengths_of_another_form_are_another_pass(stage):
    x, n = torch.randn(ROWS, COLS), torch.zeros(4, dtype=torch.int32)
    for key_len in (n[:1], n[:2], n[:1].float(), None):
        before = stage.issued()
        stage.forward(x, key_len)
        assert stage.issued() == before + 1      # through the layer code, which checks
    stage.forward(x, torch.zeros(1, dtype=torch.int32))
    assert stage.replayed() == 1


def test_forms_remembered_are_bounded(stage):
    base = torch.zeros(COLS * 64)
    for i in range(12):
        stage.forward(torch.as_strided(base, (ROWS, COLS), (COLS, 1)), torch.zeros(i + 1, dtype=torch.int32))
    assert len(stage.engine._replay.plans[("F", 1, 0)]) == replay.Replay.VARIANTS


def test_an_operand_inside_the_stages_own_buffers_is_not_recorded(stage):
    """A pointer into both could not be told apart: such a pass always goes through the layer code."""
    own = stage.module._stash[1][0][0]["out"]
    for _ in range(2):
        stage.forward(own)
        x = torch.randn(ROWS, COLS)
        stage.module._stash[1][0][0]["x0"] = x
        stage.backward(x)
    assert stage.replayed() == 0


def test_plan_operands_on_the_host(monkeypatch):
    """The native side: overlapping operands are refused, as are launches with another number of addresses."""
    with hip.Plan.record() as plan:
        pass
    a = torch.zeros(16)
    with pytest.raises(hip.HipKernelError, match="overlap"):
        plan.operands(list(map(hip.address_range, (a, a[8:]))))
    plan.operands(list(map(hip.address_range, (a[:8], a[8:], a[:0]))))
    with pytest.raises(hip.HipKernelError, match="named"):
        plan.operands([hip.address_range(a)])
    with pytest.raises(hip.HipKernelError):
        plan.launch(0, SimpleNamespace(cuda_stream=0), [a])
    with pytest.raises(hip.HipKernelError):
        hip.check(hip.lib().bb_plan_launch(plan._plan, 0, None), "bb_plan_launch")


# what a program may change between batches, and the next pass has to see
CHANGES = {
    "setting": lambda s: setattr(s.layer, "eps", 0.5),
    "new-attribute": lambda s: setattr(s.layer, "extra", 1),
    "base-seed": lambda s: setattr(s.module, "base_seed", 4),
    "weight-in-place": lambda s: s.layer.w.update(a_2=torch.ones(COLS)),
    "bind": lambda s: s.layer.bind({"a_2": torch.ones(COLS)}, {}),
    "statistics": lambda s: s.layer.running.update({1: (torch.zeros(1), torch.ones(1))}),
    "scratch": lambda s: s.ctx.scratch.update(d=torch.zeros(4)),
    "workspace": lambda s: s.ctx.ensure_workspace(1000),
    "layer": lambda s: s.module.func_buckets.update({1: [Layer(COLS)]}),
    "stash": lambda s: s.module._stash.update({1: [[{"out": torch.zeros(ROWS, COLS)}]]}),
}


@pytest.mark.parametrize("graphs", [False, True], ids=["plans", "graphs"])
@pytest.mark.parametrize("change", list(CHANGES))
def test_a_change_between_batches_reaches_the_next_pass(stage, change, graphs):
    stage.layer.w, stage.layer.running = {"a_2": torch.zeros(COLS)}, {1: (torch.zeros(1), torch.ones(1))}
    stage.engine.use_graphs = graphs
    stage.ctx.stream = SimpleNamespace(synchronize=lambda: None)
    x, g = torch.randn(ROWS, COLS), torch.randn(ROWS, COLS)
    for _ in range(3):
        stage.forward(x)
        stage.backward(g)
    assert stage.replayed() == 4
    CHANGES[change](stage)
    issued = stage.issued()
    for passes in (1, 2):
        stage.forward(x)
        stage.backward(g)
        assert stage.issued() == issued + (2 * passes if graphs else 2)      # once each; a graph is captured on the second
    stage.forward(x)
    assert stage.issued() == issued + (4 if graphs else 2) and stage.ctx.calls[-1][1] == (0.5 if change == "setting" else stage.layer.eps)


class Logging(Layer):
    def forward(self, x, st, ctx):
        return super().forward(x, st, ctx)


class Helper(Layer):
    def _scaled(self, x):
        return x


class Start(Layer):
    """Defines only how its parameters start."""

    def __init__(self, hidden):
        super().__init__(hidden)

    def init_params(self, master, seed):
        pass


class Promising(Logging):
    launches_only = True


def _shadowed():
    layer = Layer(COLS)
    layer.forward = lambda x, st, ctx: type(layer).forward(layer, x, st, ctx)
    return layer


@pytest.mark.parametrize("make,replayed", [(lambda: Logging(COLS), False), (lambda: Helper(COLS), False), (_shadowed, False), (lambda: Start(COLS), True),
                                           (lambda: Promising(COLS), False), (lambda: Layer(COLS), True)])
def test_layers_that_do_more_than_launch_are_not_replayed(stage, make, replayed):
    """Python code of a subclass, or put over a method of the object, runs in every pass; a class that promises to launch
    only has to do so for every method on the way to the promising base."""
    layer = make()
    stage.module.func_buckets[1] = [layer]
    assert replay.launches_only([layer]) == replayed
    x = torch.randn(ROWS, COLS)
    for _ in range(3):
        stage.forward(x)
    assert stage.issued() == (1 if replayed else 3)


def test_a_class_whose_passes_were_replaced_is_not_replayed(stage, monkeypatch):
    x = torch.randn(ROWS, COLS)
    stage.forward(x)
    inner = Layer.forward

    def wrapped(self, x, st, ctx):
        return inner(self, x, st, ctx)
    wrapped.__module__ = "elsewhere"
    monkeypatch.setattr(Layer, "forward", wrapped)
    for _ in range(2):
        stage.forward(x)
    assert stage.replayed() == 0 and stage.issued() == 3


class Rebuilt(Layer):
    launches_only = True

    def forward(self, x, st, ctx):
        return super().forward(x, st, ctx)

    def rebuild(self, x, st, ctx):
        pass

    def grad_sink(self, st, ctx):
        pass


def checkpointed(stage, monkeypatch):
    """The stage's passes as one checkpoint group: with the methods that only such passes call."""
    kept = torch.zeros(2, ROWS, COLS)
    monkeypatch.setattr(hip, "cast", lambda src, dst, stream=None: dst.copy_(src))
    stage.module.__dict__.update(activation_checkpoint_interval=len(stage.module.func_buckets[1]), _kept={1: [list(kept)]})
    stage.module._stash_arena[(1, "kept")] = kept


@pytest.mark.parametrize("method", replay.PASS_METHODS)
def test_a_method_of_a_pass_replaced_in_its_class_is_seen(stage, monkeypatch, method):
    """By one of the class's own module: recorded anew.  By another's: its Python code runs in every pass."""
    stage.module.func_buckets[1], n = [Rebuilt(COLS), Rebuilt(COLS)], 2
    stage.module._stash[1][0].append({"out": torch.zeros(ROWS, COLS)})
    stage.module.stage_seq[1].append(ROWS)
    if method == "rebuild":
        checkpointed(stage, monkeypatch)
    x, inner = torch.randn(ROWS, COLS), getattr(Rebuilt, method)
    stage.forward(x)
    stage.forward(x)
    assert (stage.issued(), stage.replayed()) == (n, 1)

    def other(self, *a):
        return inner(self, *a)
    monkeypatch.setattr(Rebuilt, method, other)
    for replayed in (1, 2):
        stage.forward(x)
        assert (stage.issued(), stage.replayed()) == (2 * n, replayed)

    def wrapped(self, *a):
        return inner(self, *a)
    wrapped.__module__ = "elsewhere"
    monkeypatch.setattr(Rebuilt, method, wrapped)
    for passes in (3, 4):
        stage.forward(x)
        assert (stage.issued(), stage.replayed()) == (passes * n, 2)


@pytest.mark.parametrize("method", ["forward", "backward", "_forward_into", "_rebuild"])
@pytest.mark.parametrize("where", ["class", "object"])
def test_a_method_a_pass_is_made_of_replaced_in_the_module_is_seen(stage, monkeypatch, method, where):
    x = torch.randn(ROWS, COLS)
    if method.startswith("_"):
        checkpointed(stage, monkeypatch)
    stage.forward(x)
    stage.forward(x)
    assert (stage.issued(), stage.replayed()) == (1, 1)
    target = stage.module if where == "object" else type(stage.module)
    inner = getattr(target, method)
    bound = where == "object" or method.startswith("_")
    other = (lambda *a, **kw: inner(*a, **kw)) if bound else (lambda self, *a, **kw: inner(self, *a, **kw))
    monkeypatch.setattr(target, method, staticmethod(other) if where == "class" and bound else other)
    for issued in (2, 3):
        stage.forward(x)
        assert (stage.issued(), stage.replayed()) == (issued, 1)


def test_replaying_can_be_switched_off(stage):
    x = torch.randn(ROWS, COLS)
    stage.forward(x)
    stage.engine.replay = False
    stage.forward(x)
    assert stage.replayed() == 0 and stage.issued() == 2


def test_the_frameworks_layers_promise_to_launch_only():
    from bamboo_amd import BottleNeck, DecoderLayer, FinalLayerNorm, SumLast, TransformerLayer
    from perf import cases
    layers = (TransformerLayer(64, 1, 64), DecoderLayer(64, 1, 64), FinalLayerNorm(64), SumLast(64), BottleNeck(64, 16), BottleNeck(64, 16, stride=2),
              cases._Encoder(64, 1, 64), cases._Block(64, 16))
    assert replay.launches_only(layers) and not replay.launches_only(layers + (Helper(COLS),))


def test_forgetting_gives_the_buffers_back(stage):
    """A failover replaces lanes: neither plans nor the states they were compared with keep the old one's scratch."""
    import weakref
    stage.ctx.scratch["d"] = torch.zeros(4)
    x = torch.randn(ROWS, COLS)
    stage.forward(x)
    old = weakref.ref(stage.ctx.scratch["d"])
    del stage.ctx.scratch["d"]
    assert old() is not None
    stage.engine._replay.forget()
    assert old() is None and not stage.engine._replay.plans
    stage.forward(x)
    assert stage.issued() == 2


def test_address_ranges():
    t = torch.zeros(4, 6)
    at, es = t.data_ptr(), t.element_size()
    for view, last in ((t, 23), (t[1:3], 17), (t.t(), 23), (t[:, 2:4], 21), (t[::2, 1:2], 13), (t[:1].expand(3, 6), 5)):
        assert hip.address_range(view) == (view.data_ptr(), at + (last + 1) * es)
    lo, hi = hip.address_range(t[:0])
    assert lo == hi
