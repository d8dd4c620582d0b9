"""Calls on PyTorch tensors through the native extension: the same results, checks and errors as the
general path, on the current stream, from several threads."""
import threading

import pytest
import torch

import tensorcomprehensions_amd as tc

pytestmark = pytest.mark.gpu

ADD = "def add(float(N, M) A, float(N, M) B) -> (C, D) { C(n, m) = A(n, m) + B(n, m) D(n, m) = A(n, m) - B(n, m) }"
MASK = "def mask(float(N) A, bool(N) B) -> (C) { C(n) = B(n) ? A(n) : float(0) }"


def data(n=37, m=65, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(-9, 10, (n, m), generator=g).float().cuda() for _ in range(2)]


@pytest.fixture(scope="module")
def executor():
    return tc.compile(ADD, "add", data(), "naive")


def test_the_extension_is_there_and_launches(executor):
    from tensorcomprehensions_amd import _torch_call
    A, B = data()
    outs = tc.prepare_outputs(ADD, "add", [A, B])
    plan = tc._plan(executor)
    assert isinstance(plan, _torch_call.Plan)
    assert plan.run([A, B], outs) and torch.equal(outs[0], A + B) and torch.equal(outs[1], A - B)
    assert plan.unchecked_run((B, A), tuple(outs)) and torch.equal(outs[1], B - A)
    C, D = executor(A, B)
    assert torch.equal(C, A + B) and torch.equal(D, A - B) and C.data_ptr() != outs[0].data_ptr()


@pytest.mark.parametrize("spoil", [
    lambda A, B, o: ([A], o), lambda A, B, o: ([A, B], o[:1]), lambda A, B, o: ([A, B.double()], o), lambda A, B, o: ([A, B[:, :64]], o),
    lambda A, B, o: ([A, B.cpu()], o), lambda A, B, o: ([A, B[:36]], o), lambda A, B, o: ([A, B], [o[0], o[1].int()]),
    lambda A, B, o: ([A, B], [o[0], o[1].cpu()]), lambda A, B, o: ([A, torch.empty(65, 37, device="cuda").t()], o),
])
def test_tensors_that_do_not_match_are_refused_before_any_launch(executor, spoil):
    A, B = data()
    outs = [torch.full((37, 65), 5.0, device="cuda") for _ in range(2)]
    ins, bad = spoil(A, B, outs)
    assert tc._plan(executor).run(ins, bad) is False
    with pytest.raises(tc.TcError):
        tc.run(executor, ins, bad)
    torch.cuda.synchronize()
    assert all(bool((o == 5.0).all()) for o in outs)


def test_bool_inputs_and_defined_methods_at_changing_sizes():
    T = tc.define(MASK, tc.make_naive_options_factory())
    for n in (5, 300, 5, 1):
        A = torch.arange(n, device="cuda", dtype=torch.float32)
        B = (A % 2) == 0
        assert torch.equal(T.mask(A, B), torch.where(B, A, torch.zeros_like(A)))
        assert torch.equal(T.mask(A, B.to(torch.uint8)), torch.where(B, A, torch.zeros_like(A)))
    with pytest.raises(tc.TcError):
        T.mask(A, torch.ones(7, device="cuda", dtype=torch.bool))


def test_calls_run_on_the_current_stream_and_from_threads(executor):
    A, B = data(seed=3)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        big = torch.randn(2048, 2048, device="cuda")
        for _ in range(20):
            big = big @ big * 1e-3
        A2 = A + 1.0                                # queued behind the products on the side stream
        C, _ = executor(A2, B)
        assert torch.equal(C, A2 + B)               # (compared on the same stream)
    side.synchronize()
    failures = []

    def work(seed):
        X, Y = data(seed=seed)
        with torch.cuda.stream(torch.cuda.Stream()):
            torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
            for _ in range(50):
                C, D = executor(X, Y)
            if not (torch.equal(C, X + Y) and torch.equal(D, X - Y)):
                failures.append(seed)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


def test_a_cleared_executor_reports_it():
    ex = tc.compile(ADD, "add", data(), "naive")
    A, B = data()
    ex(A, B)
    ex.clear_runtime_compiled_function()
    with pytest.raises(tc.TcError, match="No rtcFun_ attached"):
        ex(A, B)


def test_defined_methods_answer_the_same_whatever_was_called_before():
    """Strides and types that options and compilation have not seen go through them, also right after
    a call that differs in nothing else."""
    src = "def f(float(N, M) A) -> (C) { C(n, m) = A(n, m) + 1 }"
    column, row = torch.arange(5.0, device="cuda").reshape(5, 1), torch.arange(5.0, device="cuda").reshape(1, 5)
    for before in ([], [column]):
        T = tc.define(src, tc.make_naive_options_factory())
        for A in before:
            assert torch.equal(T.f(A), A + 1)
        with pytest.raises(tc.TcError, match="invalid strides"):
            T.f(row.t())                                # (5, 1) with strides (1, 5)
    asked = []

    def factory(text, entry, *inputs):
        asked.append([str(t.dtype) for t in inputs])
        return tc.MappingOptions("naive")

    T = tc.define(MASK, factory)
    A = torch.arange(8, device="cuda", dtype=torch.float32)
    B = (A % 2) == 0
    for mask in (B, B.to(torch.uint8), B):
        assert torch.equal(T.mask(A, mask), torch.where(B, A, torch.zeros_like(A)))
    assert [a[1] for a in asked] == ["torch.bool", "torch.uint8"]
