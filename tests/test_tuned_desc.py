"""The descriptor of a record is plain data: it is copied and pickled whole, with the sizes it was searched for, and made
without the library (no GPU needed)."""
import copy
import pickle

import pytest

from heron_amd import backend as B
from heron_amd import tuned


@pytest.mark.parametrize("name", ["gemm_u8s8_8192", "bmm_f16_qk", "conv2d_f16_resnet"])
def test_copies(name):
    d = tuned.load(name).desc
    for same in (copy.copy(d), copy.deepcopy(d), pickle.loads(pickle.dumps(d))):
        assert same.as_tuple() == d.as_tuple()
        assert same.tuned_for is not None and same.tuned_for == d.tuned_for


def test_made_without_the_library(monkeypatch):
    t = tuned.load("conv2d_u8s8_resnet")
    _, op, shape, dtype = tuned.CASES[t.name]
    sched, _ = tuned.instantiate(t.name, op, shape, dtype, t.records)

    def missing():
        raise RuntimeError("not built")
    monkeypatch.setattr(B, "lib", missing)
    assert sched.to_desc().as_tuple() == t.desc.as_tuple()
