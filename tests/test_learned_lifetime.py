"""A LearnedNetwork reads the pattern of the matrix given to set_graph in every
later pass, so it keeps that matrix (host only: the library call is stubbed)."""
import gc
import weakref

import kutta_amd


class Matrix:
    handle = None


class Library:
    @staticmethod
    def ka_learned_set_graph(net, matrix):
        return 0

    @staticmethod
    def ka_learned_destroy(net):
        pass


def test_network_keeps_its_matrix(monkeypatch):
    monkeypatch.setattr(kutta_amd, "host_lib", lambda: Library)
    net = kutta_amd.LearnedNetwork.__new__(kutta_amd.LearnedNetwork)
    net.handle = None
    first, second = Matrix(), Matrix()
    kept = [weakref.ref(first), weakref.ref(second)]
    net.set_graph(first)
    del first
    gc.collect()
    assert kept[0]() is not None
    net.set_graph(second)
    del second
    gc.collect()
    assert kept[0]() is None and kept[1]() is not None
