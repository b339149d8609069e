"""Losses computed by several threads at once with one network, each on its own
stream: each thread's are those it gets alone."""

import threading

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd.surrogate import UNet, pad16  # noqa: E402

DEV = "cuda:0"


def test_losses_of_threads_do_not_mix():
    net = UNet(1, 16, 7, 6, seed=1)
    n, h, w, threads, rounds = 1, 16, 64, 3, 1500
    g = torch.Generator(device=DEV).manual_seed(2)
    out = torch.randn(n * h * w * pad16(6), device=DEV, generator=g)
    targets = [10.0 ** k * torch.randn(n * h * w * 6, device=DEV, generator=g) for k in range(threads)]
    want = [net.loss_and_grad(out, t, n, h, w)[0] for t in targets]
    torch.cuda.synchronize()
    wrong = [0] * threads

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(rounds):
                wrong[k] += net.loss_and_grad(out, targets[k], n, h, w)[0] != want[k]

    ts = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert wrong == [0] * threads
    assert len(net._works) <= threads
