"""Which method fills the stash of a checkpoint group's last layer again: ``rebuild`` goes only with the ``forward`` it was cut from."""
import pytest

from bamboo_amd.layers import BottleNeck, DecoderLayer, TransformerLayer
from bamboo_amd.module import PipelineModule


class Renamed(TransformerLayer):
    pass


class OwnForward(TransformerLayer):
    def forward(self, x, st, ctx):
        return super().forward(x, st, ctx)


class OwnBoth(OwnForward):
    def forward(self, x, st, ctx):
        return super().forward(x, st, ctx)

    def rebuild(self, x, st, ctx):
        super().rebuild(x, st, ctx)


class Inherited(OwnForward):
    pass


@pytest.mark.parametrize("kind,method", [(TransformerLayer, "rebuild"), (DecoderLayer, "rebuild"), (Renamed, "rebuild"), (OwnBoth, "rebuild"),
                                         (OwnForward, "forward"), (Inherited, "forward"), (BottleNeck, "forward")])
def test_rebuild_goes_with_its_forward(kind, method):
    layer = object.__new__(kind)
    assert PipelineModule._rebuild(layer) == getattr(layer, method)
    layer.forward = lambda x, st, ctx: None      # one put over it on the object
    assert PipelineModule._rebuild(layer) is layer.forward


def test_output_goes_where_it_is_kept():
    """The stash's ``out`` is the kept buffer during the call and itself again afterwards, also after an error; where shapes differ, or the
    layer has no such entry, it is left alone."""
    import torch

    class Layer:
        def forward(self, x, st, ctx):
            self.seen = st.get("out")
            if ctx == "fail":
                raise RuntimeError("no")
            return self.seen

    layer, own, kept = Layer(), torch.zeros(4, 8), torch.zeros(4, 8)
    st = {"out": own}
    assert PipelineModule._forward_into(kept, layer, None, st, None) is kept and st["out"] is own
    with pytest.raises(RuntimeError):
        PipelineModule._forward_into(kept, layer, None, st, "fail")
    assert st["out"] is own
    for other in ({"out": torch.zeros(4, 4)}, {"out": own.double()}, {}):
        PipelineModule._forward_into(kept, layer, None, dict(other), None)
        assert layer.seen is other.get("out")
