"""Times of a kernel's launches, for tests of the rules that choose between two kernels."""
import torch


def graph_us(call, launches=20, replays=12):
    """The least time of a launch in a captured chain of them, in microseconds."""
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(launches):
            call()
    times = []
    for _ in range(replays):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        graph.replay()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b))
    return min(times) * 1e3 / launches
