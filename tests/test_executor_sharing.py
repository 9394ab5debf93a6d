"""What the networks of a process share -- pinned blocks, the record of who is open and who has run -- without a device: networks are
built bare, on a stand-in for the library."""
import gc
import threading

from armnn_amd.executor import DeviceNetwork


class FakeLibrary:
    """Pinned memory that only counts."""

    def __init__(self):
        self.live, self.allocated, self.freed = set(), 0, 0

    def mi355x_host_alloc(self, p, nbytes):
        self.allocated += 1
        p._obj.value = self.allocated << 24
        self.live.add(p._obj.value)
        return 0

    def mi355x_host_free(self, p):
        self.live.remove(p)
        self.freed += 1
        return 0


class FakeDevice:
    def stream_destroy(self, s):
        pass


def bare_network(lib, lanes=1):
    n = object.__new__(DeviceNetwork)
    n.lib, n.dev, n.stream, n.lanes = lib, FakeDevice(), 1, lanes
    n.graphs, n.chains, n.tails, n.plans, n.buffers, n._side_streams = {}, [], [], [], {}, None
    n._register()
    return n


class Owner:
    """As a program's own class around a network: closes it when it is collected, which a reference cycle leaves to the garbage
    collector, at whatever allocation of whatever thread that runs."""

    def __init__(self, network):
        self.network, self.cycle = network, self

    def __del__(self):
        self.network.close()


def test_close_from_a_garbage_collection_inside_the_sharing_code():
    lib = FakeLibrary()
    keeper = bare_network(lib, lanes=2)
    done = threading.Event()
    threshold = gc.get_threshold()

    def work():
        for allocations in range(1, 120):                  # the collection runs at each of them in turn
            gc.disable()
            gc.collect()
            for _ in range(3):
                n = bare_network(lib, lanes=2)
                n._one_lane_now()
                n._give_blocks(n._take_blocks(2))
                Owner(n)
            del n
            gc.set_threshold(gc.get_count()[0] + allocations)
            gc.enable()
            other = bare_network(lib, lanes=2)
            keeper._one_lane_now()
            keeper._give_blocks(keeper._take_blocks(3))
            other._one_lane_now()
            other.close()
        done.set()

    thread = threading.Thread(target=work, daemon=True)
    try:
        thread.start()
        assert done.wait(20), "the sharing code waits for itself"
    finally:
        gc.set_threshold(*threshold)
        gc.enable()
    thread.join()
    gc.collect()
    keeper.close()
    assert not lib.live                                    # nothing is kept once the last network is closed


def test_repeated_calls_allocate_no_pinned_memory():
    """The largest call takes a block for each of its parts and one for the results; two networks may be in a call at once."""
    lib = FakeLibrary()
    a, b = bare_network(lib), bare_network(lib)
    for _ in range(3):
        a._give_blocks(a._take_blocks(DeviceNetwork._MOST_PARTS + 1))
        assert (lib.allocated, lib.freed) == (33, 0)
    for _ in range(3):
        first, second = a._take_blocks(20), b._take_blocks(20)
        assert not set(first) & set(second)
        a._give_blocks(first)
        b._give_blocks(second)
        assert (lib.allocated, lib.freed) == (40, 0)
    b.close()
    assert len(lib.live) == 33                             # what one network's call takes
    a.close()
    assert not lib.live
