"""KV tiers on CPU: host offload + reload after HBM eviction, disk spill, remote cache
server sharing between two engines, controller reporting, P->D page push, serde."""

import asyncio
import copy
import gc
import threading
import weakref

import numpy as np
import pytest
import torch

from vllm_production_stack_amd import ops
from vllm_production_stack_amd.cache_server import CacheServer
from vllm_production_stack_amd.engine.config import EngineConfig, KVOffloadConfig, KVTransferConfig
from vllm_production_stack_amd.engine.llm_engine import LLMEngine
from vllm_production_stack_amd.engine.request import SamplingParams
from vllm_production_stack_amd.kv.remote import RemoteKVClient
from vllm_production_stack_amd.kv.serde import PageSerde, rc_decode, rc_encode

SP = SamplingParams(max_tokens=4, temperature=0, ignore_eos=True)


LAYOUT = {"groups": 1}


@pytest.fixture(autouse=True, params=[1, 2], ids=["whole-pages", "layer-groups"])
def pool_layout(request):
    """Every test here runs on a pool of whole pages and on one pool per layer (tiny-llama has two
    layers): the lower tiers see the same flat page either way."""
    LAYOUT["groups"] = request.param
    yield
    LAYOUT["groups"] = 1


def engine(pages=24, **off):
    cfg = EngineConfig(model="tiny-llama", device="cpu", dtype="float32", max_model_len=1024,
                       max_num_seqs=8, max_num_batched_tokens=256, num_gpu_blocks_override=pages,
                       kv_offload=KVOffloadConfig(**off), kv_layer_groups=LAYOUT["groups"], port=0)
    return LLMEngine(cfg)


def prompts(n, length, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(16, 500, (length,), generator=g).tolist() for _ in range(n)]


def test_range_coder_roundtrip_and_gain():
    rng = np.random.default_rng(0)
    sym = np.clip(np.round(rng.normal(0, 3, 200000)), -15, 15).astype(np.int8)
    blob = rc_encode(sym, 50000, 4)
    assert len(blob) < 0.5 * sym.size  # ~3.6 bits of entropy per symbol
    assert np.array_equal(rc_decode(blob, sym.size, 50000, 4), sym)
    wide = rng.integers(-127, 128, 10000).astype(np.int8)
    assert np.array_equal(rc_decode(rc_encode(wide, 0, 1), wide.size, 0, 1), wide)


def test_page_serde_naive_and_cachegen():
    n_layers, n_kv, hd = 3, 1, 128
    page = torch.randn(n_layers * 2 * n_kv * 64 * hd).to(torch.bfloat16)
    naive = PageSerde(n_layers, n_kv, hd, torch.bfloat16, "naive")
    assert torch.equal(naive.decode(naive.encode(page), torch.device("cpu")), page)
    cg = PageSerde(n_layers, n_kv, hd, torch.bfloat16, "cachegen", levels=[127, 31, 15])
    blob = cg.encode(page)
    assert len(blob) < 0.5 * page.numel() * 2
    back = cg.decode(blob, torch.device("cpu")).float()
    x = page.float()
    first = slice(0, 2 * n_kv * 64 * hd)
    assert (x[first] - back[first]).abs().mean() / x[first].abs().mean() < 0.03
    assert (x - back).abs().mean() / x.abs().mean() < 0.15


def test_damaged_page_blobs_are_refused_not_decoded():
    """Blobs come back from disk and from other hosts: a cut, padded or corrupted one has to be
    a ValueError (the tier code turns that into a cache miss), never a page of wrong values."""
    import pytest

    n_layers, n_kv, hd = 3, 1, 128
    page = torch.randn(n_layers * 2 * n_kv * 64 * hd).to(torch.bfloat16)
    with pytest.raises(ValueError):
        rc_decode(rc_encode(np.zeros(50000, np.int8) + 3, 0, 1)[:10], 50000, 0, 1)
    with pytest.raises(ValueError):
        rc_decode(b"", 100, 0, 1)
    for kind in ("naive", "cachegen"):
        sd = PageSerde(n_layers, n_kv, hd, torch.bfloat16, kind, levels=[127, 31, 15])
        blob = sd.encode(page)
        sd.decode(blob, torch.device("cpu"))
        for bad in (b"", blob[:7], blob[:len(blob) // 2], blob[:-1], blob + b"x", b"\x00" * len(blob),
                    blob[:4] + b"\xff" * 8 + blob[12:]):
            with pytest.raises(ValueError):
                sd.decode(bad, torch.device("cpu"))
            with pytest.raises(ValueError):
                sd.unpack(bad)
    other = PageSerde(n_layers + 1, n_kv, hd, torch.bfloat16, "naive")
    with pytest.raises(ValueError):
        other.decode(blob, torch.device("cpu"))


def test_rans_reference_roundtrip_and_gain():
    """NumPy definition of the GPU entropy stage: exact round trip on Gaussian, constant and
    uniform contexts, output close to the zeroth-order entropy."""
    from vllm_production_stack_amd.ops import reference as ref

    rng = np.random.default_rng(1)
    n_ctx, spc, ctx_len = 4, 256, 256 * 128
    sym = np.clip(np.round(rng.normal(0, 5, n_ctx * ctx_len)), -128, 127).astype(np.int8)
    sym[ctx_len:2 * ctx_len] = -3                                        # one symbol only
    sym[2 * ctx_len:3 * ctx_len] = rng.integers(-128, 128, ctx_len)      # incompressible
    freq, states, sizes, coded = ref.rans_encode(sym, n_ctx, spc)
    assert freq.shape == (n_ctx, 256) and (freq.astype(int).sum(1) == 4096).all()
    assert sizes.astype(int).sum() == coded.size and sizes.max() <= 2 * ctx_len // spc
    back = ref.rans_decode(freq, states, sizes, coded, sym.size, n_ctx, spc)
    assert np.array_equal(back.view(np.int8), sym)
    first = sym[:ctx_len].view(np.uint8)
    p = np.bincount(first, minlength=256) / ctx_len
    entropy_bytes = -(p[p > 0] * np.log2(p[p > 0])).sum() * ctx_len / 8
    assert sizes[:spc].astype(int).sum() < 1.03 * entropy_bytes
    assert sizes[spc:2 * spc].astype(int).sum() == 0                     # a constant context costs nothing


def test_page_serialiser_can_be_copied_and_pickled():
    import pickle

    page = torch.randn(3 * 2 * 2 * 64 * 64).to(torch.bfloat16)
    cg = PageSerde(3, 2, 64, torch.bfloat16, "cachegen", levels=[127, 31, 15])
    for twin in (copy.deepcopy(cg), pickle.loads(pickle.dumps(cg))):
        assert twin.encode(page) == cg.encode(page)


def test_cachegen_rans_payload_restores_like_the_range_coder():
    """Serde kind 2 (quantiser + rANS) read back on a CPU-only host equals kind 1 of the same page."""
    n_layers, n_kv, hd = 3, 1, 128
    torch.manual_seed(5)
    page = torch.randn(n_layers * 2 * n_kv * 64 * hd).to(torch.bfloat16)
    cg = PageSerde(n_layers, n_kv, hd, torch.bfloat16, "cachegen", levels=[127, 31, 15])
    via_range_coder = cg.decode(cg.encode(page), torch.device("cpu"))
    lv = torch.tensor(cg.levels, dtype=torch.int32)
    from vllm_production_stack_amd import ops
    sym, scales = ops.cachegen_encode(page, lv, cg.unit_elems, n_layers)
    blob = cg.pack(cg.rans_payload(sym, scales), None)
    assert cg.unpack(blob)[0] == "rans"
    assert torch.equal(cg.decode(blob, torch.device("cpu")), via_range_coder)
    assert torch.equal(cg.restore(cg.unpack(blob), torch.device("cpu")), via_range_coder)
    assert len(blob) < 0.6 * page.numel() * 2
    with pytest.raises(ValueError):
        cg.decode(blob[:-100], torch.device("cpu"))


def test_host_offload_survives_hbm_eviction():
    eng = engine(pages=12, local_cpu=True, max_local_cpu_gb=0.05)
    a, b, c = prompts(3, 330)
    first = eng.generate([a], copy.deepcopy(SP))[0]
    # two more long prompts push a's pages out of the 12-page HBM pool
    eng.generate([b], copy.deepcopy(SP))
    eng.generate([c], copy.deepcopy(SP))
    r = eng.add_request(a, copy.deepcopy(SP))
    while eng.has_work():
        eng.step()
    # the 5 full pages are back: the head page(s) may have survived in HBM, the rest came from host
    assert r.num_cached_tokens + r.num_external_tokens == 320 and r.num_external_tokens >= 192
    assert r.output_ids == first
    assert eng.connector.host.loads >= 3


def test_disk_tier_after_host_eviction(tmp_path):
    eng = engine(pages=12, local_cpu=True, max_local_cpu_gb=0.0000001, max_local_disk_gb=0.1,
                 local_disk_path=str(tmp_path))
    assert eng.connector.host.n_slots == 1  # host tier keeps a single page: everything spills
    a, b = prompts(2, 330, seed=1)
    first = eng.generate([a], copy.deepcopy(SP))[0]
    eng.generate([b], copy.deepcopy(SP))
    eng.generate(prompts(1, 330, seed=2), copy.deepcopy(SP))
    r = eng.add_request(a, copy.deepcopy(SP))
    while eng.has_work():
        eng.step()
    assert r.num_cached_tokens + r.num_external_tokens == 320 and r.num_external_tokens >= 192
    assert r.output_ids == first
    assert len(list(tmp_path.rglob("*.kv"))) > 0  # under the model-identity directory


def test_pages_on_disk_are_the_same_for_both_pool_layouts(tmp_path):
    """A replica with one pool per layer writes its pages to disk; a replica with whole pages (and
    the other way round) finds them there and continues with the same tokens."""
    mine = LAYOUT["groups"]
    a = prompts(1, 330, seed=9)[0]
    writer = engine(pages=12, max_local_disk_gb=0.1, local_disk_path=str(tmp_path))
    first = writer.generate([a], copy.deepcopy(SP))[0]
    assert len(getattr(writer.runner.pool, "groups", [0])) == mine
    writer.shutdown()
    LAYOUT["groups"] = 3 - mine
    reader = engine(pages=12, max_local_disk_gb=0.1, local_disk_path=str(tmp_path))
    assert len(getattr(reader.runner.pool, "groups", [0])) == 3 - mine
    r = reader.add_request(a, copy.deepcopy(SP))
    while reader.has_work():
        reader.step()
    assert r.num_external_tokens == 320 and r.output_ids == first


def _serve_in_thread(coro_factory):
    loop = asyncio.new_event_loop()
    box = {}

    def run():
        asyncio.set_event_loop(loop)
        box["obj"] = loop.run_until_complete(coro_factory())
        box["ready"].set()
        loop.run_forever()

    box["ready"] = threading.Event()
    t = threading.Thread(target=run, daemon=True)
    t.start()
    box["ready"].wait(10)
    return loop, box["obj"]


class _Device:
    """A device whose copies are over only when somebody waits: stands in for the calls of ``PageSerde.decode`` on a GPU, and notes
    pinned buffers that go back to their allocator while a copy still reads them."""

    def __init__(self, monkeypatch, fail=False):
        self.queued, self.over, self.early, self.buffers, self.fail = 0, 0, 0, 0, fail
        self.lock, self.all_in, self.reads = threading.RLock(), None, {}
        empty, dev = torch.empty, self

        class Event:
            def record(self, stream=None):
                self.at = dev.queued

            def synchronize(self):
                dev.over = max(dev.over, self.at)

        class Stream:
            def synchronize(self):
                dev.over = dev.queued

        def pinned_empty(*size, pin_memory=False, **kw):
            t = empty(*size, **kw)
            if pin_memory:
                with dev.lock:
                    dev.buffers += 1
                    key = dev.buffers
                t.key = key
                weakref.finalize(t, dev.freed, key)
            return t

        def page_decode(src, pinned, size, n, n_ctx, unit_elems, device, spc=ops.RANS_SPC):
            with dev.lock:
                dev.queued += 1
                dev.reads[pinned.key] = dev.queued
            if dev.all_in is not None:
                dev.all_in.wait(20)
            if dev.fail:
                raise RuntimeError("cachegen_decode: unsupported arguments")
            return empty(n, dtype=torch.bfloat16)

        monkeypatch.setattr(torch, "empty", pinned_empty)
        monkeypatch.setattr(torch.cuda, "Event", Event)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: Stream())
        monkeypatch.setattr(ops, "page_decode", page_decode)

    def freed(self, key):
        self.early += self.reads.get(key, 0) > self.over


def _rans_blob(monkeypatch):
    sd = PageSerde(3, 2, 64, torch.bfloat16, "cachegen", levels=[31, 31, 15])
    sym, scales = ops.cachegen_encode(torch.randn(sd.page_elems).bfloat16(), torch.tensor(sd.levels, dtype=torch.int32), sd.unit_elems, 3)
    return sd, sd.pack(sd.rans_payload(sym, scales), None)


@pytest.mark.parametrize("callers", [1, 2, 3, 5])
def test_pinned_buffers_outlive_the_copies_that_read_them(callers, monkeypatch):
    """More callers at once than a serialiser keeps buffers, and a serialiser that ends with copies still queued."""
    sd, blob = _rans_blob(monkeypatch)
    dev = _Device(monkeypatch)
    dev.all_in = threading.Barrier(callers)
    threads = [threading.Thread(target=sd.decode, args=(blob, torch.device("cuda"))) for _ in range(callers)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(30)
    gc.collect()
    assert dev.queued == callers and dev.buffers == callers and dev.early == 0
    dev.all_in = None
    sd.decode(blob, torch.device("cuda"))
    del sd, threads, t
    gc.collect()
    assert dev.early == 0 and dev.over == dev.queued


def test_pinned_buffers_outlive_a_call_that_fails(monkeypatch):
    sd, blob = _rans_blob(monkeypatch)
    dev = _Device(monkeypatch, fail=True)
    for _ in range(4):
        with pytest.raises(RuntimeError):
            sd.decode(blob, torch.device("cuda"))
    gc.collect()
    assert dev.queued == 4 and dev.early == 0


@pytest.mark.parametrize("serde", ["naive", "cachegen"])
def test_remote_cache_shared_between_engines(serde):
    loop, srv = _serve_in_thread(lambda: CacheServer("127.0.0.1", 0, 1 << 30).start())
    url = f"lm://127.0.0.1:{srv.port}"
    try:
        e1 = engine(remote_url=url, remote_serde=serde)
        e2 = engine(remote_url=url, remote_serde=serde)
        (a,) = prompts(1, 330, seed=3)
        first = e1.generate([a], copy.deepcopy(SP))[0]
        import time

        for _ in range(50):
            if RemoteKVClient(url).stats().get("keys", 0) >= 5:
                break
            time.sleep(0.05)
        r = e2.add_request(a, copy.deepcopy(SP))
        while e2.has_work():
            e2.step()
        assert r.num_external_tokens == 320  # e2 never computed this prompt
        if serde == "naive":
            assert r.output_ids == first
        else:
            assert len(r.output_ids) == 4
        e1.shutdown()
        e2.shutdown()
    finally:
        asyncio.run_coroutine_threadsafe(srv.stop(), loop).result(10)
        loop.call_soon_threadsafe(loop.stop)


def test_remote_page_evicted_between_store_and_reload_is_a_cache_miss():
    """The cache server is a bounded LRU: pages this replica uploaded can be gone when it wants
    them back.  That is a cache miss (recompute from the first missing page), not an error, and
    the HBM pages reserved for the load are given back."""
    probe = engine()
    page_bytes = probe.runner.page_bytes
    probe.shutdown()
    # room for about two pages: every further upload evicts the oldest one
    loop, srv = _serve_in_thread(lambda: CacheServer("127.0.0.1", 0, int(2.5 * page_bytes)).start())
    url = f"lm://127.0.0.1:{srv.port}"
    try:
        eng = engine(pages=12, remote_url=url, remote_serde="naive")
        free0 = eng.bm.num_free()
        a, b, c = prompts(3, 330, seed=7)
        first = eng.generate([a], copy.deepcopy(SP))[0]
        eng.generate([b], copy.deepcopy(SP))
        eng.generate([c], copy.deepcopy(SP))  # a's pages are out of HBM, most are out of the server too
        import time

        time.sleep(0.3)  # let the background uploads (and the evictions they cause) finish
        r = eng.add_request(a, copy.deepcopy(SP))
        while eng.has_work():
            eng.step()  # must not raise
        assert r.output_ids == first
        assert r.num_cached_tokens + r.num_external_tokens < 320  # something had to be recomputed
        assert eng.bm.num_free() == free0  # no page leaked by the failed load
        eng.shutdown()
    finally:
        asyncio.run_coroutine_threadsafe(srv.stop(), loop).result(10)
        loop.call_soon_threadsafe(loop.stop)


def test_remote_server_gone_is_a_cache_miss():
    loop, srv = _serve_in_thread(lambda: CacheServer("127.0.0.1", 0, 1 << 30).start())
    url = f"lm://127.0.0.1:{srv.port}"
    eng = engine(pages=12, remote_url=url, remote_serde="naive")
    a, b, c = prompts(3, 330, seed=9)
    first = eng.generate([a], copy.deepcopy(SP))[0]
    eng.generate([b], copy.deepcopy(SP))
    eng.generate([c], copy.deepcopy(SP))
    asyncio.run_coroutine_threadsafe(srv.stop(), loop).result(10)
    loop.call_soon_threadsafe(loop.stop)
    r = eng.add_request(a, copy.deepcopy(SP))
    while eng.has_work():
        eng.step()
    assert r.output_ids == first and r.num_external_tokens == 0
    eng.shutdown()


def test_two_models_on_one_cache_server_do_not_share_pages():
    """Same tokenizer, same KV geometry, different weights identity: the chain hashes of a prompt
    are equal, the keys in the shared server are not."""
    loop, srv = _serve_in_thread(lambda: CacheServer("127.0.0.1", 0, 1 << 30).start())
    url = f"lm://127.0.0.1:{srv.port}"
    try:
        def eng_named(name):
            cfg = EngineConfig(model="tiny-llama", served_model_name=name, device="cpu", dtype="float32",
                               max_model_len=1024, max_num_seqs=8, max_num_batched_tokens=256,
                               num_gpu_blocks_override=24,
                               kv_offload=KVOffloadConfig(remote_url=url, remote_serde="naive"), port=0)
            return LLMEngine(cfg)

        e1, e2, e3 = eng_named("base"), eng_named("fine-tune"), eng_named("base")
        assert e1.connector.namespace != e2.connector.namespace == e2.connector.namespace
        assert e1.connector.namespace == e3.connector.namespace
        (a,) = prompts(1, 330, seed=11)
        e1.generate([a], copy.deepcopy(SP))
        import time

        for _ in range(50):
            if RemoteKVClient(url).stats().get("keys", 0) >= 5:
                break
            time.sleep(0.05)
        r2 = e2.add_request(a, copy.deepcopy(SP))
        while e2.has_work():
            e2.step()
        assert r2.num_external_tokens == 0  # another model's pages are invisible
        r3 = e3.add_request(a, copy.deepcopy(SP))
        while e3.has_work():
            e3.step()
        assert r3.num_external_tokens == 320  # a replica of the same model finds them
        for e in (e1, e2, e3):
            e.shutdown()
    finally:
        asyncio.run_coroutine_threadsafe(srv.stop(), loop).result(10)
        loop.call_soon_threadsafe(loop.stop)


@pytest.mark.parametrize("api_key", [None, "sekret"])
def test_controller_reporting_and_pd_push(api_key):
    from vllm_production_stack_amd.controller import KVController, start_controller
    from vllm_production_stack_amd.engine.async_engine import AsyncLLMEngine
    from vllm_production_stack_amd.engine.block_manager import chain_hashes
    from vllm_production_stack_amd.engine.server import serve

    ctrl = KVController()
    loop, runner = _serve_in_thread(lambda: start_controller(ctrl, "127.0.0.1", 0))
    cport = runner.addresses[0][1]

    async def go():
        dec_cfg = EngineConfig(model="tiny-llama", device="cpu", dtype="float32", max_model_len=1024,
                               num_gpu_blocks_override=32, host="127.0.0.1", api_key=api_key,
                               kv_transfer=KVTransferConfig("LMCacheConnectorV1", "kv_consumer"))
        dec = LLMEngine(dec_cfg)
        dae = AsyncLLMEngine(dec)
        dae.start(asyncio.get_running_loop())
        drunner = await serve(dae, "127.0.0.1", 0)
        dport = drunner.addresses[0][1]
        pre_cfg = EngineConfig(model="tiny-llama", device="cpu", dtype="float32", max_model_len=1024,
                               num_gpu_blocks_override=32, host="127.0.0.1", port=1, api_key=api_key,
                               kv_transfer=KVTransferConfig("LMCacheConnectorV1", "kv_producer"),
                               kv_offload=KVOffloadConfig(enable_controller=True, instance_id="prefill-0",
                                                          controller_url=f"127.0.0.1:{cport}"))
        pre = LLMEngine(pre_cfg)
        (a,) = prompts(1, 330, seed=4)

        def run_prefill():
            sp = SamplingParams(max_tokens=1, temperature=0, ignore_eos=True)
            req = pre.add_request(a, sp, kv_transfer_params={"do_remote_decode": True,
                                                             "decode_target": f"http://127.0.0.1:{dport}"})
            while pre.has_work():
                pre.step()
            # the step loop did not wait for the transfer: it runs on the push worker, and the
            # request's HTTP handler would await this future before answering the router
            fut = pre.connector.push_future(req.request_id)
            assert fut is not None and pre.connector.push_future(req.request_id) is None
            assert fut.result(30)["mode"] == "tcp"
            pre.idle_tick()  # the references the worker held on the pages are given back
            assert pre.bm.num_free() == 32

        await asyncio.get_running_loop().run_in_executor(None, run_prefill)
        # decode replica now holds the prompt's 5 full pages without having computed them
        assert dec.bm.peek_prefix(chain_hashes(a)) == 5
        out = []
        async for so in dae.generate("d1", a, copy.deepcopy(SP)):
            out.extend(so.new_token_ids)
            cached = so.num_cached_tokens
        assert cached == 320
        ref = engine().generate([a], copy.deepcopy(SP))[0]
        assert out == ref
        for _ in range(50):
            if ctrl.lookup(chain_hashes(a)):
                break
            await asyncio.sleep(0.05)
        assert ctrl.lookup(chain_hashes(a)) == {"prefill-0": 320}
        assert ctrl.query_instance("127.0.0.1") == "prefill-0"
        await drunner.cleanup()
        dae.stop()
        pre.shutdown()

    try:
        asyncio.run(go())
    finally:
        asyncio.run_coroutine_threadsafe(runner.cleanup(), loop).result(10)
        loop.call_soon_threadsafe(loop.stop)


def test_prefix_caching_off_with_host_tier_serves_every_turn_from_host():
    """``--no-enable-prefix-caching`` + CPU offload (the reference's benchmark configuration): HBM
    keeps nothing between requests, a repeated prompt is loaded from the host tier."""
    cfg = EngineConfig(model="tiny-llama", device="cpu", dtype="float32", max_model_len=1024,
                       max_num_seqs=8, max_num_batched_tokens=256, num_gpu_blocks_override=24,
                       enable_prefix_caching=False,
                       kv_offload=KVOffloadConfig(local_cpu=True, max_local_cpu_gb=0.05), port=0)
    eng = LLMEngine(cfg)
    (a,) = prompts(1, 330, seed=21)
    first = eng.generate([a], copy.deepcopy(SP))[0]
    assert eng.bm.num_free() == 24 and not eng.bm.cached  # nothing stays in HBM
    for _ in range(2):
        r = eng.add_request(a, copy.deepcopy(SP))
        while eng.has_work():
            eng.step()
        assert r.output_ids == first
        assert r.num_cached_tokens == 0 and r.num_external_tokens == 320
    assert eng.connector.host.loads >= 10
    eng.shutdown()


@pytest.mark.parametrize("prefix_caching", [False, True])
def test_pages_filled_by_a_requests_last_token_are_offloaded_while_still_owned(prefix_caching):
    """A request whose last computed token fills a page finishes in the step that fills it.  The
    offload copy takes a reference on that page, which is only worth something while the request
    still owns the page: taken after the request had handed the page back, it landed on a free
    page, the next request was given that page with a fresh count of one, and the copy's release
    freed it under the new owner (two requests writing one page; later a negative count)."""
    cfg = EngineConfig(model="tiny-llama", device="cpu", dtype="float32", max_model_len=1024,
                       max_num_seqs=8, max_num_batched_tokens=256, num_gpu_blocks_override=24,
                       enable_prefix_caching=prefix_caching,
                       kv_offload=KVOffloadConfig(local_cpu=True, max_local_cpu_gb=0.05), port=0)
    eng = LLMEngine(cfg)
    seen = []
    orig = eng.connector.store_pages

    def spy(fresh):
        seen.append([eng.bm.ref[p] for _, p in fresh])
        eng.bm.pin([p for _, p in fresh])  # what an asynchronous copy does ...
        eng.bm.free([p for _, p in fresh])  # ... and what its completion does
        return orig(fresh)

    eng.connector.store_pages = spy
    sp = SamplingParams(max_tokens=5, temperature=0, ignore_eos=True)
    # 60 prompt tokens + 4 computed output tokens = 64: the page fills in the step that samples the 5th
    for seed in (31, 32, 33):
        eng.generate(prompts(1, 60, seed=seed), copy.deepcopy(sp))
    assert len(seen) == 3 and all(r and min(r) > 0 for r in seen), seen
    assert eng.bm.num_free() == 24 and all(c == 0 for c in eng.bm.ref)
    assert len(set(eng.bm.free_ids)) == len(eng.bm.free_ids)  # no page is on the free list twice
    eng.shutdown()


def test_a_free_page_cannot_be_pinned():
    from vllm_production_stack_amd.engine.block_manager import BlockManager

    bm = BlockManager(4)
    (p,) = bm.allocate(1)
    bm.pin([p])
    bm.free([p])
    assert bm.ref[p] == 1 and p not in bm.free_ids  # the reader's reference keeps it
    bm.free([p])
    assert p in bm.free_ids
    with pytest.raises(AssertionError, match="is free"):
        bm.pin([p])
    # a cached page waiting for eviction can be pinned and leaves the eviction list for that time
    (q,) = bm.allocate(1)
    bm.register(q, 1234)
    bm.free([q])
    assert q in bm.evictable
    bm.pin([q])
    assert q not in bm.evictable and bm.ref[q] == 1
    bm.free([q])
    assert q in bm.evictable


def test_staged_download_returns_its_slots_when_the_connection_dies_half_way():
    """Bulk download of raw pages through the pinned staging ring: a cache server that stops
    answering after k pages must not cost the ring a single slot (a leaked slot per hiccup would
    end with the engine thread blocked on an empty ring), and a ring that stays empty makes the
    download fall back to the per-page path instead of waiting for ever."""
    import queue

    import torch

    from vllm_production_stack_amd.kv.connector import KVConnector

    elems, n_slots = 64, 4

    class Serde:
        page_elems = elems

        def _header(self, n):
            return b"HDR" + int(n).to_bytes(4, "little")

    class Remote:
        def __init__(self, die_after):
            self.calls, self.die_after = 0, die_after

        def get_page_into(self, key, hdr_len, view):
            self.calls += 1
            if self.calls > self.die_after:
                raise ConnectionError("server went away")
            view[:] = bytes([self.calls]) * len(view)
            return Serde()._header(elems * 2)

    c = object.__new__(KVConnector)
    c.device = torch.device("cpu")
    c.serde = Serde()
    c._stage = torch.zeros((n_slots, elems), dtype=torch.bfloat16)
    c._stage_free = queue.Queue()
    for i in range(n_slots):
        c._stage_free.put(i)
    c.pool = torch.zeros((16, elems), dtype=torch.bfloat16)
    c._key = lambda h: f"k{h}"
    c.remote = Remote(die_after=6)  # more pages than slots: the ring is recycled once, then the link dies
    items = [(100 + i, i) for i in range(10)]
    with pytest.raises(ConnectionError):
        c._download_staged(items)
    assert c._stage_free.qsize() == n_slots
    # pages that did arrive are in the pool
    assert bool((c.pool[0].view(torch.uint8) == 1).all()) and bool((c.pool[5].view(torch.uint8) == 6).all())
    # an exhausted ring (uploads hold every slot): the rest is handed to the per-page path
    held = [c._stage_free.get() for _ in range(n_slots)]
    c.remote = Remote(die_after=100)
    c.STAGE_WAIT_S = 0.05
    assert c._download_staged(items[:3]) == items[:3]
    for sl in held:
        c._stage_free.put(sl)
    assert c._download_staged(items[:3]) == [] and c._stage_free.qsize() == n_slots
