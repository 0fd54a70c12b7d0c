"""The logits of recorded steps: what a caller holds stays what it was when the next steps run."""
import pytest
import torch

from configs import TINY

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
B, STEPS = 5, 7


def _echo():
    from xinfer_amd.parts import Head

    class Echo(Head):
        graph_safe = True

        def forward(self, h):
            return h
    return Echo


def _view():
    from xinfer_amd.parts import Head

    class View(Head):
        graph_safe = True

        def forward(self, h):
            return h[:, ::2]
    return View


def _kept():
    from xinfer_amd.parts import Head

    class Kept(Head):
        graph_safe = True
        buf = None

        def forward(self, h):
            if self.buf is None or self.buf.shape != h.shape:
                self.buf = torch.empty(h.shape, dtype=torch.float32, device=h.device)
            self.buf.copy_(h)
            return self.buf
    return Kept


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("head", [None, _echo, _view, _kept])
def test_logits_that_are_held(head, dtype, model_dirs):
    """All rows and some rows of recorded steps, held to the end, are bit for bit those of the same steps launched kernel by kernel: with the built-in head, and
    with heads that return their input, a view of it, or a buffer of their own that they write again."""
    from xinfer_amd.engine import ModelRunner, StepEntry, load_model
    model = load_model(model_dirs["B"], dtype, DEV)
    if head is not None:
        model.head = head()(model.head.spec, model.dtype)

    def run(use_graphs):
        runner = ModelRunner(model, TINY["B"]["page_size"], 8 * B, B, use_graphs=use_graphs, graph_after=1)
        for i in range(B):
            runner.add_request(i)
        runner.step([StepEntry(i, [3 + i, 40 + i], []) for i in range(B)])
        held = []
        for step in range(STEPS):
            wanted = [i for i in range(B) if step % 2 == 0 or i % 3 == 1]
            y = runner.step([StepEntry(i, [(7 * step + i) % 50], [0] if i in wanted else []) for i in range(B)])
            held.append(y if use_graphs and step > 0 else y.clone())       # (the first one records: it runs launch by launch)
        return [y.clone() for y in held], runner.graph_replays

    want, none = run(False)
    got, replays = run(True)
    assert none == 0 and replays == STEPS - 1
    for step, (a, b) in enumerate(zip(want, got)):
        assert a.shape == b.shape and torch.equal(a, b), f"step {step}"
