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
