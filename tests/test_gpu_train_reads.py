"""What a program reads of a learning net: weights below, at and above the sizes that are copied through page-locked memory, from
one thread and from several at once, are the ones the net was given; and a loss and weights after learning do not depend on
how they are read."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
# floats: one, 1024 and one row more (the smallest that come through), 131072 (the largest) and one row more
SIZES = [(1, 1), (16, 64), (17, 64), (256, 512), (257, 512)]


@pytest.mark.parametrize("O,K", SIZES)
def test_weights_come_back_as_given(O, K):
    from n2d2_amd import frame_hip
    rng = np.random.default_rng(O * 1000 + K)
    net = frame_hip.TrainNet(rng.random((2, K, 1, 1), dtype=np.float32), propagate_gradient=False)
    w = rng.standard_normal((O, K)).astype(np.float32)
    net.add_fc("fc", w)
    for _ in range(3):
        assert np.array_equal(net.weights("fc"), w)


def test_several_threads_read_one_net():
    from n2d2_amd import frame_hip
    rng = np.random.default_rng(7)
    net = frame_hip.TrainNet(rng.random((2, 300, 1, 1), dtype=np.float32), propagate_gradient=False)
    given, last = {}, 300
    for i, O in enumerate((70, 400, 33, 8)):
        given["fc%d" % i] = rng.standard_normal((O, last)).astype(np.float32)
        net.add_fc("fc%d" % i, given["fc%d" % i])
        last = O
    wrong = []

    def read(name):
        for _ in range(50):
            if not np.array_equal(net.weights(name), given[name]):
                wrong.append(name)

    threads = [threading.Thread(target=read, args=(n,)) for n in given for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("batch", [2, 5])
def test_learning_again_uses_the_targets_of_the_call(batch):
    """Each learn() copies its targets without a wait: two nets, one learning A then B, the other B after its state was brought
    to the same point by A, come to the same loss and weights whatever array the targets were in."""
    from n2d2_amd import frame_hip
    rng = np.random.default_rng(batch)
    x, w = rng.random((batch, 48, 1, 1), dtype=np.float32), rng.standard_normal((40, 48)).astype(np.float32)
    a, b = (rng.random((batch, 40, 1, 1), dtype=np.float32) for _ in range(2))
    got = []
    for reuse in (False, True):
        net = frame_hip.TrainNet(x, propagate_gradient=False)
        net.add_fc("fc", w)
        net.add_softmax("softmax")
        t = np.empty_like(a)
        losses = []
        for k, v in enumerate((a, b, a, b)):
            if reuse:
                t[...] = v
                losses.append(net.learn(t, 1 + k))
                t[...] = -1.0
            else:
                losses.append(net.learn(v.copy(), 1 + k))
        got.append((losses, net.weights("fc")))
    assert got[0][0] == got[1][0] and np.array_equal(got[0][1], got[1][1])
    # no iteration: no loss, nothing changes
    before = net.weights("fc")
    assert net.learn(a, 0) == 0.0 and np.array_equal(before, net.weights("fc"))
