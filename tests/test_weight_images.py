"""The weight images that the modules keep (_PackedWeights) are those of the weights as they are: not of others
that came to lie at the same address with the same version, type and shape."""
import copy
import gc
import pickle

import numpy as np
import pytest
import torch

from gpt_triton_amd import gpt


def tensor_over(memory, shape=(4, 4)):
    """A tensor with a storage of its own over this memory: what a freed weight's address handed out again
    is to the next weight."""
    return torch.from_numpy(np.frombuffer(memory, dtype=np.float32)).view(shape)


def image(weight):
    return weight.clone()


def refill(memory, value):
    memory[:] = np.full(16, value, dtype=np.float32).tobytes()


@pytest.mark.parametrize("how", ["another parameter", "another parameter, the first alive", "its data twice"])
def test_another_weight_at_the_same_address(how):
    images, memory = gpt._PackedWeights(), bytearray(64)
    param = torch.nn.Parameter(tensor_over(memory), requires_grad=False)
    first = param
    assert torch.equal(images.get("w", param, image), torch.zeros(4, 4))
    if how == "its data twice":
        param.data = torch.ones(4, 4)
        refill(memory, 3.0)
        param.data = tensor_over(memory)
    else:
        if how == "another parameter":
            del first, param
            gc.collect()
        refill(memory, 3.0)
        param = torch.nn.Parameter(tensor_over(memory), requires_grad=False)
    assert param._version == 0
    assert images.held("w", param) is None
    assert torch.equal(images.get("w", param, image), torch.full((4, 4), 3.0))


def test_another_order_of_the_same_storage():
    images = gpt._PackedWeights()
    param = torch.nn.Parameter(torch.arange(16.0).view(4, 4), requires_grad=False)
    images.get("w", param, image)
    param.data = param.data.t()
    assert images.held("w", param) is None


def test_the_same_weight_keeps_its_image_and_no_weight_is_kept_alive():
    images = gpt._PackedWeights()
    param = torch.nn.Parameter(torch.zeros(4, 4), requires_grad=False)
    hit = images.get("w", param, image)
    assert images.get("w", param, image) is hit and images.held("w", param) is hit
    param.add_(1)  # in place: the version counts on
    assert images.held("w", param) is None
    assert torch.equal(images.get("w", param, image), torch.ones(4, 4))
    images.clear()
    assert images.held("w", param) is None
    images.get("w", param, image)
    storage = torch.multiprocessing.reductions.StorageWeakRef(param.untyped_storage())
    del param
    gc.collect()
    assert storage.expired()


def test_modules_with_images_are_copied_and_pickled_without_them():
    mlp = gpt.FusedMLP(64).eval()
    mlp._packed.get("ffn1_weight", mlp.ffn1_weight, image)
    for other in (copy.deepcopy(mlp), pickle.loads(pickle.dumps(mlp))):
        assert torch.equal(other.ffn1_weight, mlp.ffn1_weight)
        assert other._packed is not mlp._packed
        assert other._packed.held("ffn1_weight", other.ffn1_weight) is None
    del other
    gc.collect()
    assert mlp._packed.held("ffn1_weight", mlp.ffn1_weight) is not None
    # the state that a module pickled by an earlier version of this class brings
    images = gpt._PackedWeights.__new__(gpt._PackedWeights)
    images.__setstate__({"_entries": {"ffn1_weight": (0, 0, torch.float32, (64, 256), None)}})
    assert images.held("ffn1_weight", mlp.ffn1_weight) is None
