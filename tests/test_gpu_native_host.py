"""The native host side of an attention call away from the ordinary call: other streams,
captured graphs and several threads, without a workspace and with one."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = {"one": ([700], 16, 8), "few": ([128, 2000, 900, 1, 513], 16, 8),
          "many rows": ([300 + 7 * i for i in range(40)], 16, 8),
          # a table of three rounds: 16 rows and 24, both sides of the rule for a side stream;
          # 128, 120 and 136, both sides of the rule for counters at hand
          "two": ([700, 768], 16, 8), "three": ([700, 768, 513], 16, 8),
          "sixteen": ([768 - 40 * i for i in range(16)], 16, 8),
          "fifteen": ([768 - 40 * i for i in range(15)], 16, 8),
          "seventeen": ([768 - 40 * i for i in range(17)], 16, 8)}


def _layer(name, seed, dtype=torch.bfloat16):
    from nanovllm_jax_amd import Attention, create_decode_context
    lens, heads, kv_heads = SHAPES[name]
    bs, dev, n = 64, "cuda:0", len(lens)
    pages = [-(-x // bs) for x in lens]
    g = torch.Generator(device=dev).manual_seed(seed)
    order = np.random.default_rng(seed).permutation(sum(pages))
    table = np.full((n, max(pages)), -1, np.int32)
    ends = np.cumsum(pages)
    for b, (e, p) in enumerate(zip(ends, pages)):
        table[b, :p] = order[e - p:e]
    slots = [table[b, (x - 1) // bs] * bs + (x - 1) % bs for b, x in enumerate(lens)]
    attn = Attention(heads, 128, 128 ** -0.5, kv_heads, bs)
    rand = lambda *shape: torch.randn(shape, generator=g, device=dev).to(dtype)
    attn.set_kv_cache(*(rand(sum(pages), bs, kv_heads, 128) for _ in range(2)))
    up = lambda a: torch.from_numpy(np.asarray(a, np.int32)).to(dev)
    context = create_decode_context(up(lens), up(slots), up(table))
    args = rand(n, heads, 128), rand(n, kv_heads, 128).float(), rand(n, kv_heads, 128), context
    return attn, args


def _two_launches(attn, args):
    """The general path: the store and the attention behind each other."""
    from nanovllm_jax_amd import paged_attention, store_kv_to_cache
    q, k, v, c = args
    kc, vc = attn.k_cache.clone(), attn.v_cache.clone()
    store_kv_to_cache(k, v, kc, vc, c.slot_mapping)
    return paged_attention(q, kc, vc, c.block_tables, c.context_lens, attn.scale,
                           attn.block_size), kc, vc


def _check(attn, out, want):
    torch.testing.assert_close(out.float(), want[0].float(), rtol=1e-2, atol=2e-3)
    assert torch.equal(attn.k_cache, want[1]) and torch.equal(attn.v_cache, want[2])


@pytest.mark.parametrize("name", SHAPES)
def test_call_on_a_side_stream_and_in_a_graph_without_a_workspace(name):
    print(f"case side stream {name}", flush=True)
    attn, args = _layer(name, 3)
    want = _two_launches(attn, args)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        outs = [attn(*args) for _ in range(3)]
    torch.cuda.synchronize()
    for out in outs:
        _check(attn, out, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = attn(*args)
    for _ in range(4):
        captured.zero_()
        attn.k_cache.view(-1, 8, 128)[args[3].slot_mapping.long()] = 0
        graph.replay()
        torch.cuda.synchronize()
        _check(attn, captured, want)
        _check(attn, attn(*args), want)           # the program's own work in between


@pytest.mark.parametrize("streams", ["null", "own"])
def test_calls_of_several_threads(streams):
    """Several threads, each a layer of its own: on the null stream, whose counters they share
    in turn, or each on a stream of its own."""
    print(f"case threads on {streams} stream", flush=True)
    from nanovllm_jax_amd.layers.paged_attention import DecodeWorkspace
    layers = [_layer(name, 10 + i) for i, name in enumerate(SHAPES)]
    wants = [_two_launches(*layer) for layer in layers]
    if streams == "own":                     # one of them with a workspace
        q, _, _, c = layers[1][1]
        layers[1][0].workspace = DecodeWorkspace.for_shape(
            q.shape[0], q.shape[1], 128, c.block_tables.shape[1], 64, 8, "cuda:0")
    torch.cuda.synchronize()
    results, errors = [[] for _ in layers], []

    def work(i):
        try:
            stream = torch.cuda.Stream() if streams == "own" else torch.cuda.default_stream()
            with torch.cuda.stream(stream):
                for _ in range(50):
                    results[i].append(layers[i][0](*layers[i][1]))
            stream.synchronize()
        except Exception as e:              # noqa: BLE001 (reported by the main thread)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(layers))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for (attn, _), want, outs in zip(layers, wants, results):
        assert len(outs) == 50
        for out in outs:
            _check(attn, out, want)


def test_other_threads_run_while_a_call_enqueues():
    """Nothing but a call that gives the interpreter up lets a second thread run here: the
    time after which the interpreter would be taken from this one is set out of reach."""
    print("case interpreter released", flush=True)
    import sys
    import time
    attn, args = _layer("one", 5)
    attn(*args)
    torch.cuda.synchronize()
    ticks, stop, interval = [0], [False], sys.getswitchinterval()

    def count():
        while not stop[0]:
            ticks[0] += 1
            time.sleep(0)

    thread = threading.Thread(target=count)
    try:
        sys.setswitchinterval(100.0)     # (in front of the first wait of the other thread)
        thread.start()
        before = ticks[0]
        for _ in range(400):
            attn(*args)
        seen = ticks[0] - before
    finally:
        sys.setswitchinterval(interval)
        stop[0] = True
    thread.join()
    print("ran", seen, "times in 400 calls", flush=True)
    assert seen > 10      # (once or twice: something else gave it up)
