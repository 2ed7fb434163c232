"""A partition is an ordinary object: it can be referred to weakly, carries what a caller attaches to it, and the function makes what the class's own call does."""
import copy
import gc
import weakref

import pytest
import torch


@pytest.mark.parametrize("make", ["partition", "Partition"])
def test_weak_references_and_attributes_of_a_caller(fake_hip, make):
    p = getattr(fake_hip, make)(torch.zeros(4, 8), [2, 8])
    gone = []
    watch = weakref.ref(p, gone.append)
    p.label = "logits"
    assert watch() is p and vars(p)["label"] == "logits" and copy.copy(p).label == "logits"
    fake_hip.saxpy(fake_hip.partition(torch.zeros(64), [64]), 0.5, torch.zeros(64))
    del p
    gc.collect()
    assert gone == [watch]


def test_the_function_makes_what_the_class_does(fake_hip):
    ct, t = fake_hip, torch.zeros(4, 8)
    for shape, *rest in (([2, 8],), ((2, 8), True), ([4, 4], False, ct.U32)):
        a, b = ct.partition(t, shape, *rest), ct.Partition(t, list(shape), *rest)
        assert type(a) is type(b) and vars(a) == vars(b) and a.tensor is t
