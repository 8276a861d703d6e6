"""A call owns the plans it was given until it returns, whatever becomes of the list they came in."""
import collections.abc
import sys
import threading

import pytest
import torch

import protenix_amd as P
from protenix_amd import native
from oracle import pairformer_oracle as O
from tests.util import oracle_and_product


class Key(str):
    """A parameter's name whose look-up can be watched (a plan is examined by looking its parameters up)."""
    seen = None

    def __hash__(self):
        if Key.seen is not None:
            Key.seen()
        return str.__hash__(self)

    def __eq__(self, other):
        return str.__eq__(self, other)


def test_plans_outlive_the_sequence_they_came_in():
    ln = P.FusedLayerNorm(8)
    weight = ln._parameters.pop("weight")
    ln._parameters[Key("weight")] = weight

    def plan():
        return native.host().Plan(native._guard(ln))
    kept = plan()

    class Handed(collections.abc.Sequence):        # nobody else holds what it hands out
        def __len__(self):
            return 3

        def __getitem__(self, i):
            if i >= 3:
                raise IndexError
            return plan()
    held = []
    Key.seen = lambda: held.append(sys.getrefcount(weight))
    try:
        assert native.host().first_stale([kept]) == -1 and len(held) == 1
        alone = held.pop()
        assert native.host().first_stale(Handed()) == -1
    finally:
        Key.seen = None
    assert max(held) == alone + 3       # all three records hold the parameter while they are examined


@pytest.mark.gpu
def test_a_stack_called_by_two_threads_while_its_parameters_change():
    """A parameter is replaced between calls by equal values, so that every call finds some plans stale and all
    results are the same."""
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=4)
    s, z, pm = (t.cuda() for t in O.make_inputs(40, n_pad=3))
    with torch.no_grad():
        s0, z0 = prod(s, z, pm)
    torch.cuda.synchronize()
    wrong, lock = [], threading.Lock()

    def work(k):
        with torch.no_grad():
            for i in range(12):
                lin = prod.blocks[(i + k) % 4].tri_mul_in.linear_g
                with lock:
                    lin.weight = torch.nn.Parameter(lin.weight.detach())
                s1, z1 = prod(s, z, pm)
                if not (torch.equal(s1, s0) and torch.equal(z1, z0)):
                    wrong.append((k, i))
    ts = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong


@pytest.mark.gpu
def test_a_recording_outlives_the_plans_it_was_made_with():
    """A parameter replaced by equal values makes the plan stale; the eager call that follows makes another, and the
    memory of the first must still be the recording's."""
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=2)
    s, z, pm = (t.cuda() for t in O.make_inputs(40, n_pad=3))
    fast = P.Graphed(prod)
    s0, z0 = fast(s, z, pm)
    with torch.no_grad():
        for b in prod.blocks:
            b.tri_mul_in.linear_g.weight = torch.nn.Parameter(b.tri_mul_in.linear_g.weight.detach())
        prod(s, z, pm)
        torch.cuda.synchronize()
        junk = [torch.full((n,), float("nan"), device="cuda") for n in (98304, 131072, 1 << 20, 1 << 21, 1 << 22) for _ in range(4)]
        for _ in range(2):
            s1, z1 = fast(s, z, pm)
            assert bool(torch.equal(s1, s0)) and bool(torch.equal(z1, z0))
    del junk


@pytest.mark.gpu
def test_a_plan_made_on_one_stream_and_used_on_another():
    """The weights are still to be laid out when the second stream's call is issued, and the plan goes away while
    that call may still read them."""
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=3)
    s, z, pm = (t.cuda() for t in O.make_inputs(40, n_pad=3))
    mul = prod.blocks[0].tri_mul_out
    with torch.no_grad():
        s0, z0 = prod(s, z, pm)
        u0 = mul(z, pm)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        native._plans.clear()
        torch.cuda.synchronize()
        with torch.no_grad():
            with torch.cuda.stream(a):
                torch.cuda._sleep(20_000_000)       # (some 10 ms, then the weights)
                prod(s, z, pm)
                mul(z, pm)
            with torch.cuda.stream(b):
                s1, z1 = prod(s, z, pm)
                u1 = mul(z, pm)
                native._plans.clear()               # (the weights' memory goes back)
            with torch.cuda.stream(a):
                torch.full((4_000_000,), float("nan"), device="cuda")
        torch.cuda.synchronize()
        assert bool(torch.equal(s1, s0)) and bool(torch.equal(z1, z0)) and bool(torch.equal(u1, u0))
