"""Which calls of the GravNet block take its layers together: decided on the host, checked here without a GPU."""
import torch

from hgcalml_amd import RaggedGravNet


def block(**kwargs):
    return RaggedGravNet(13, 9, 3, 30, 11, **kwargs)


def test_compiled_blocks_trace_through_the_question():
    """a compiler that traces the block reaches its search without a break: the question is answered inside the graph"""
    layer = block()

    def question(x):
        return x + 1 if layer._layers_in_one_pass(x) else x - 1
    x = torch.randn(20, 13)
    assert torch.equal(torch.compile(question, fullgraph=True, backend="eager")(x), x - 1)


def test_replacements_are_called(monkeypatch):
    """a method or forward replaced on the instance or on the class, as a tracer or a user's own variant does it: only the layers
    one by one call it"""
    from hgcalml_amd import GravNetLayersRagged as module
    monkeypatch.setattr(module, "_library_takes", lambda *tensors: True)  # no GPU here
    layer, linear, x = block(), block(feature_activation="linear"), torch.randn(20, 13)
    assert layer._layers_in_one_pass(x) and linear._layers_in_one_pass(x)
    for name in ("compute_neighbours_and_distancesq", "collect_neighbours", "create_output_features"):
        with monkeypatch.context() as m:
            m.setattr(RaggedGravNet, name, lambda *args: None)
            assert not layer._layers_in_one_pass(x), name
        own = block()
        setattr(own, name, lambda *args: None)
        assert not own._layers_in_one_pass(x), name
    for cls in (module.TallLinear, torch.nn.ReLU, torch.nn.Identity):
        with monkeypatch.context() as m:
            m.setattr(cls, "forward", lambda self, x: x)
            taken = layer._layers_in_one_pass(x), linear._layers_in_one_pass(x)
        assert taken == (cls is torch.nn.Identity, cls is torch.nn.ReLU), cls
    assert layer._layers_in_one_pass(x) and linear._layers_in_one_pass(x)
