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
    """Streams, events and graphs that only note what was asked of them; an event is done when the test says so."""

    def __init__(self):
        self.handles, self.log, self.done = 0, [], set()

    def stream(self):
        self.handles += 1
        return self.handles

    event = stream

    def event_done(self, e):
        return e in self.done

    def event_destroy(self, e):
        self.log.append(("event_destroy", e))

    def graph_end(self, stream):
        return self.stream()

    def __getattr__(self, name):
        return lambda *a: self.log.append((name,) + a)


def bare_network(lib, lanes=1, dev=None):
    n = object.__new__(DeviceNetwork)
    n.lib, n.dev, n.stream, n.lanes, n.use_graph = lib, dev or FakeDevice(), 1, lanes, True
    n.steps = [("layer", lambda stream, lane=0, lanes=1: n.dev.log.append(("launch", lane, lanes)))]
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


def test_a_pass_runs_as_one_lane_only_while_another_networks_pass_is_under_way():
    """What networks that are merely open have done before does not matter."""
    lib, dev = FakeLibrary(), FakeDevice()
    a, b, c = (bare_network(lib, lanes=2, dev=dev) for _ in range(3))

    def passes(network):
        """Lanes that a pass of the network replays a graph for."""
        dev.log.clear()
        network.enqueue()
        return [e[0] for e in dev.log].count("graph_launch")

    assert passes(a) == 2 and passes(a) == 2               # by itself, again and again
    assert passes(b) == 1                                  # a's pass is under way
    dev.done.update((a._pass_end._event, b._pass_end._event))
    assert passes(c) == 2                                  # a and b are open, have run, and are idle
    assert passes(a) == 1
    dev.done.add(a._pass_end._event)
    assert passes(c) == 2
    c.close()
    dev.done.discard(b._pass_end._event)
    assert passes(a) == 1
    b.close()
    assert passes(a) == 2
    a.close()


def test_only_the_first_pass_captures():
    lib, dev = FakeLibrary(), FakeDevice()
    a, b = (bare_network(lib, lanes=2, dev=dev) for _ in range(2))
    a.enqueue()
    assert [e[1:] for e in dev.log if e[0] == "launch"] == [(0, 2), (1, 2), (0, 1)]
    b.enqueue()
    dev.log.clear()
    for _ in range(2):
        a.enqueue()                                        # as one lane: b's pass is under way
        b.close()
    assert not [e for e in dev.log if e[0] in ("launch", "graph_begin")]
    a.close()
