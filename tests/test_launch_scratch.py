"""Scratch that several launches of one call share: who may come between them, and what runs without it.

On the host, with a HIP runtime that records launches (fake_hip.py).
"""
from __future__ import annotations

import pytest

from tests.fake_hip import fake_hip  # noqa: F401  (fixture)

# Calls of two and more launches over the scratch of their stream.
CALLS = {
    "attention of several tokens": "lambda: attention(64, 1000)",
    "attention of one token": "lambda: attention(1, 4000)",
    "integer linear": "lambda: lib.lh_linear(C.byref(weight(8, 256, 2048, 128)), buffer.ptr, 64, 8, buffer.ptr, None, None)",
}


@pytest.mark.parametrize("first", CALLS)
@pytest.mark.parametrize("second", ["attention of several tokens", "integer linear"])
def test_two_threads_on_one_stream(fake_hip, first, second):  # noqa: F811
    # every call's launches follow each other: another thread's call would
    # overwrite what the first of them left for the last
    runs = fake_hip(f"""
        fake.fake_set_launch_delay_us(300)
        calls = [{CALLS[first]}, {CALLS[second]}]
        lengths = []
        for call in calls:
            assert call() == 0
            lengths.append(len(kernels()))
        gate = threading.Barrier(2)
        def work(call):
            gate.wait()
            for _ in range(20): assert call() == 0
        threads = [threading.Thread(target=work, args=(call,)) for call in calls]
        for t in threads: t.start()
        for t in threads: t.join()
        runs = []                                    # [thread, launches in a row]
        for entry in log():
            if entry[0] != "launch": continue
            if runs and runs[-1][0] == entry[1]: runs[-1][1] += 1
            else: runs.append([entry[1], 1])
        per = {{}}
        for thread, n in runs: per.setdefault(thread, []).append(n)
        # a thread's calls all have one length: its runs are multiples of it
        result = [sorted(lengths), sorted([sum(v) // 20, all(n % (sum(v) // 20) == 0 for n in v)] for v in per.values())]
    """)
    lengths, threads = runs
    assert lengths[0] >= 2 and [n for n, _ in threads] == lengths
    assert all(whole for _, whole in threads)


def test_captured_attention_keeps_no_scratch(fake_hip):  # noqa: F811
    # A graph may be launched on another stream, beside this stream's own
    # calls: several tokens run unsplit in it, also where scratch is there.
    eager, captured, per_thread = fake_hip("""
        stream = rt.Stream()
        assert attention(64, 1000, stream=stream.handle) == 0
        eager = kernels()
        fake.fake_set_capturing(1)
        assert attention(64, 1000, stream=stream.handle) == 0
        captured = kernels()
        assert attention(64, 1000) == 0              # on the null stream, which may not be asked then
        captured += kernels()
        fake.fake_set_capturing(0)
        # one handle for every thread's own default stream
        assert attention(64, 1000, stream=2) == 0
        result = eager, captured, kernels()
    """)
    assert len(eager) == 2 and "merge" in eager[1]
    assert len(captured) == 2 and all("attention_rows_kernel" in k for k in captured)
    assert len(per_thread) == 1 and "attention_rows_kernel" in per_thread[0]


def test_attention_without_memory_for_scratch(fake_hip):  # noqa: F811
    # splitting the keys is a choice: a call that finds no memory for it runs
    # unsplit, and splits again once there is some
    statuses, short, later = fake_hip("""
        fake.fake_set_malloc_limit(1 << 16)
        statuses = [attention(64, 1000), attention(64, 1000)]
        short = kernels()
        fake.fake_set_malloc_limit(1 << 40)
        statuses.append(attention(64, 1000))
        result = statuses, short, kernels()
    """)
    assert statuses == [0, 0, 0]
    assert len(short) == 2 and all("attention_rows_kernel" in k for k in short)
    assert len(later) == 2 and "merge" in later[1]


def test_unaligned_quantized_input(fake_hip):  # noqa: F811
    # copied to where the faster GEMMs can load it, except into a graph or
    # where there is no memory: a kernel takes it as it is
    result = fake_hip("""
        stream = rt.Stream()
        def call(group): return lib.lh_linear_q(C.byref(weight(8, 256, 2048, group)), buffer.ptr + 4, buffer.ptr, 64,
                                                buffer.ptr, None, stream.handle)
        def what(): return [e[0] if e[0] == "copy" else e[2] for e in log()]
        result = []
        for group in (128, 2048):
            assert call(group) == 0
            eager = what()
            fake.fake_set_capturing(1)
            assert call(group) == 0
            captured = what()
            fake.fake_set_capturing(0)
            result.append([eager, captured])
        fake.fake_set_malloc_limit(1 << 21)
        big = lambda: lib.lh_linear_q(C.byref(weight(8, 64, 2048, 128)), buffer.ptr + 4, buffer.ptr, 1000, buffer.ptr,
                                      None, stream.handle)
        result.append([big(), what()])
    """)
    for eager, captured in result[:2]:
        assert eager[0] == "copy" and "gemm" in eager[1]
        assert len(captured) == 1 and "gemm_grouped_kernel" in captured[0] and "Lb0E" in captured[0]
    status, launched = result[2]
    assert status == 0 and len(launched) == 1 and "Lb0E" in launched[0]


PRESETS = {"qwen": (14, 2, 64), "smollm2": (15, 5, 64), "heads of 128": (32, 8, 128)}


@pytest.mark.parametrize("shape", PRESETS)
def test_prompts_share_their_keys_as_layer_calls_do(fake_hip, shape, tmp_path):  # noqa: F811
    # a session's scratch is enough for every prompt length and position: its
    # attention launches the grids of the layer call, which allocates what it needs
    heads, kv, dim = PRESETS[shape]
    wrong, split = fake_hip(f"""
        from dataclasses import replace
        from leaf_amd import artifact, models
        spec = models.PRESETS["smollm2"](reduced=True)
        spec = replace(spec, hidden={heads * dim}, layers=1, heads={heads}, kv_heads={kv}, head_dim={dim}, max_positions=4096)
        path = sys.argv[2] + "/one.leaf"
        artifact.write_artifact(path, spec, seed=1)
        decoder = rt.Decoder(path, 32, max_context=4096, max_prefill=512)
        def grids(): return [e[2:3] + e[4:] for e in log() if e[0] == "launch" and "attention" in e[2]]
        wrong, split = [], 0
        for tokens in (2, 3, 5, 16, 33, 64, 100, 191, 256, 400, 511, 512):
            for position in (0, 1, 63, 150, 700, 1500, 2500, 3584):
                decoder.reset()
                done = 0
                while done < position:
                    n = min(512, position - done)
                    decoder.forward_into(np.zeros(n, np.uint32), None)
                    done += n
                log()
                decoder.forward_into(np.zeros(tokens, np.uint32), None)
                session = grids()
                assert attention(tokens, position, {heads}, {kv}, {dim}) == 0
                if session != grids(): wrong.append([tokens, position])
                split += len(session) == 2
        result = wrong, split
    """, str(tmp_path))
    assert wrong == [] and split >= 40


def test_session_without_memory_for_partial_results(fake_hip, tmp_path):  # noqa: F811
    launched = fake_hip("""
        from leaf_amd import artifact, models
        path = sys.argv[2] + "/tiny.leaf"
        artifact.write_artifact(path, models.PRESETS["qwen"](reduced=True), seed=1)
        fake.fake_set_malloc_limit(5 << 20)              # the model and its workspaces fit, 9 MB of partial results do not
        decoder = rt.Decoder(path, 32, max_context=512, max_prefill=256)
        log()
        decoder.forward_into(np.zeros(200, np.uint32), None)
        result = [k for k in kernels() if "attention" in k]
    """, str(tmp_path))
    assert len(launched) == 2 and all("attention_rows_kernel" in k for k in launched)    # one a layer
