"""Loading checkpoints onto the GPU (reference: MiracleModel.from_pretrained,
model.py:58-72; weights.py:14-99, 145-208; config.py:100-117) and the command
line over HIP (cli.py:30-95).

The workload geometries are written to disk as a BF16 safetensors bundle, a
sharded index and a native-name npz (with a native config.json whose family is
auto-detected); each must load with ``from_pretrained`` into a model whose
logits equal, bit for bit, those of the same weights handed over in memory.
"""
import json

import numpy as np
import pytest

from miracle_hip import MiracleModel, ModelConfig, presets, synthetic
from miracle_hip.cli import main
from miracle_hip.weights import BF16Array, SafeTensors, native_names, write_safetensors

pytestmark = pytest.mark.gpu

IDS = [3, 141, 59, 26, 535, 89, 79, 323, 846, 264, 338, 327]


def _write_bundle(directory, config, weights):
    directory.mkdir()
    (directory / "config.json").write_text(json.dumps(config.to_dict()))
    write_safetensors(directory / "model.safetensors", weights)


@pytest.fixture(scope="module")
def mid():
    wl = presets.workload("flashnano-1.5-mid")
    return ModelConfig.from_dict(wl["config"]), synthetic.synthetic_weights(wl["config"], wl["seed"], wl["dtype"])


def test_bundle_and_shards_load_bit_exact(backend, tmp_path, mid):
    config, weights = mid
    with MiracleModel(config, weights, backend=backend, context_length=64) as model:
        want = model.prefill(IDS, return_all=True)
        stream = model.generate(IDS, max_new_tokens=4)
    _write_bundle(tmp_path / "bundle", config, weights)
    assert SafeTensors(tmp_path / "bundle" / "model.safetensors").entries["layers.0.q"][1] == "BF16"
    with MiracleModel.from_pretrained(tmp_path / "bundle", backend=backend, context_length=64) as loaded:
        assert loaded.weight_cache.resident == 2 * sum(v.bits.size for v in weights.values()
                                                       if isinstance(v, BF16Array)) + \
            4 * sum(np.asarray(v).size for v in weights.values() if not isinstance(v, BF16Array))
        np.testing.assert_array_equal(loaded.prefill(IDS, return_all=True), want)
    # the same tensors over three shards and an index
    shards = tmp_path / "sharded"
    shards.mkdir()
    (shards / "config.json").write_text(json.dumps(config.to_dict()))
    names = list(weights)
    parts = [names[i::3] for i in range(3)]
    weight_map = {}
    for i, part in enumerate(parts):
        write_safetensors(shards / f"part-{i}.safetensors", {k: weights[k] for k in part})
        weight_map.update({k: f"part-{i}.safetensors" for k in part})
    (shards / "model.safetensors.index.json").write_text(json.dumps({"weight_map": weight_map}))
    with MiracleModel.from_pretrained(shards, backend=backend, context_length=64) as loaded:
        np.testing.assert_array_equal(loaded.prefill(IDS, return_all=True), want)
    # the command line on the bundle
    assert main(["generate", str(tmp_path / "bundle"), "--ids", " ".join(map(str, IDS)), "--max-new-tokens", "4",
                 "--context-length", "64"]) == 0


def test_cli_generate_and_devices(backend, tmp_path, mid, capsys):
    config, weights = mid
    with MiracleModel(config, weights, backend=backend, context_length=64) as model:
        stream = model.generate(IDS, max_new_tokens=5)
        sampled = model.generate(IDS, max_new_tokens=5, temperature=0.7, top_k=20, top_p=0.9, seed=3)
    _write_bundle(tmp_path / "bundle", config, weights)
    capsys.readouterr()
    assert main(["generate", str(tmp_path / "bundle"), "--ids", ",".join(map(str, IDS)), "--max-new-tokens", "5",
                 "--context-length", "64"]) == 0
    out = json.loads(capsys.readouterr().out)
    assert out["token_ids"] == stream and out["device"]["arch"].startswith("gfx950")
    assert main(["generate", str(tmp_path / "bundle"), "--ids", ",".join(map(str, IDS)), "--max-new-tokens", "5",
                 "--context-length", "64", "--temperature", "0.7", "--top-k", "20", "--top-p", "0.9",
                 "--seed", "3"]) == 0
    assert json.loads(capsys.readouterr().out)["token_ids"] == sampled
    assert main(["devices"]) == 0
    devices = json.loads(capsys.readouterr().out)
    assert devices and all(d["arch"].startswith("gfx950") for d in devices)
    assert main(["generate", str(tmp_path / "bundle"), "--ids", "999999", "--context-length", "64"]) == 2
    assert "vocabulary" in capsys.readouterr().err


@pytest.mark.parametrize("case", ["native_15", "native_16", "native_17", "native_heavy", "native_lighting",
                                  "native_lite"])
def test_native_npz_with_native_config_loads_bit_exact(backend, golden_dir, tmp_path, case):
    """A checkpoint under the training repository's names with a native
    config.json (the reference's own native configs; the family is detected
    from their keys) loads like the weights handed over in memory."""
    native_config = json.loads((golden_dir / "configs.json").read_text())[case]["input"]
    config = ModelConfig.from_dict(native_config)
    weights = synthetic.micro_weights(config)
    names = native_names(config)
    directory = tmp_path / case
    directory.mkdir()
    np.savez(directory / "model.npz", **{names[k]: v for k, v in weights.items()})
    (directory / "config.json").write_text(json.dumps(native_config))
    ids = [i % config.vocab_size for i in IDS[:6]]
    with MiracleModel(config, weights, backend=backend, context_length=16) as model:
        want = model.prefill(ids, return_all=True)
    with MiracleModel.from_pretrained(directory, backend=backend, context_length=16) as loaded:
        assert loaded.config == config
        np.testing.assert_array_equal(loaded.prefill(ids, return_all=True), want)


def test_exported_bundles_load_on_the_gpu(backend, tmp_path, mid):
    """Export (reference export.py:41-80) of the flashnano-1.5 mid workload
    from a native-name PyTorch BF16 state dict and from a native-name npz: the
    BF16-keeping bundle loads with from_pretrained into a model whose logits
    equal the in-memory model's bit for bit; the widened FP32 bundle (the
    reference's own format) runs the FP32-weight kernels on the same values,
    so its logits agree within the BF16 tolerance and its greedy stream is the
    same.  The command line's export writes the same bundle."""
    torch = pytest.importorskip("torch")
    from miracle_hip.export import export_checkpoint
    config, weights = mid
    with MiracleModel(config, weights, backend=backend, context_length=64) as model:
        want = model.prefill(IDS, return_all=True)
        stream = model.generate(IDS, max_new_tokens=4)
    names = native_names(config)
    state = {}
    for key, value in weights.items():
        if isinstance(value, BF16Array):
            state[names[key]] = torch.from_numpy(value.bits.view(np.int16)).view(torch.bfloat16)
        else:
            state[names[key]] = torch.from_numpy(np.asarray(value, np.float32))
    torch.save({"model_state_dict": state}, tmp_path / "ckpt.pt")
    (tmp_path / "config.json").write_text(json.dumps(config.to_dict()))
    print("case export torch state dict -> BF16 bundle", flush=True)
    assert export_checkpoint(tmp_path / "ckpt.pt", tmp_path / "config.json", tmp_path / "bf16") == config
    assert SafeTensors(tmp_path / "bf16" / "model.safetensors").entries["layers.0.q"][1] == "BF16"
    with MiracleModel.from_pretrained(tmp_path / "bf16", backend=backend, context_length=64) as loaded:
        np.testing.assert_array_equal(loaded.prefill(IDS, return_all=True), want)
        assert loaded.generate(IDS, max_new_tokens=4) == stream
    print("case export widened FP32 bundle (command line)", flush=True)
    assert main(["export", "--checkpoint", str(tmp_path / "ckpt.pt"), "--config", str(tmp_path / "config.json"),
                 "--output", str(tmp_path / "f32"), "--fp32"]) == 0
    assert SafeTensors(tmp_path / "f32" / "model.safetensors").entries["layers.0.q"][1] == "F32"
    with MiracleModel.from_pretrained(tmp_path / "f32", backend=backend, context_length=64) as loaded:
        np.testing.assert_allclose(loaded.prefill(IDS, return_all=True), want, rtol=1e-3, atol=1e-4)
        assert loaded.generate(IDS, max_new_tokens=4) == stream
    print("case export native npz (FP32 values) -> bundle", flush=True)
    del state
    native = tmp_path / "native"
    native.mkdir()
    np.savez(native / "model.npz", **{names[k]: np.asarray(v, np.float32) for k, v in weights.items()})
    assert export_checkpoint(native / "model.npz", tmp_path / "config.json", tmp_path / "npz") == config
    assert SafeTensors(tmp_path / "npz" / "model.safetensors").entries["layers.0.q"][1] == "F32"
    with MiracleModel.from_pretrained(tmp_path / "npz", backend=backend, context_length=64) as loaded:
        np.testing.assert_allclose(loaded.prefill(IDS, return_all=True), want, rtol=1e-3, atol=1e-4)
        assert loaded.generate(IDS, max_new_tokens=4) == stream


def test_freed_buffers_are_recycled_within_bounds():
    """Buffers freed by tensors serve later tensors of their size, hold at most
    the pool's bytes, and go back to the library when an allocation fails."""
    from miracle_hip import HIPBackend, HIPError
    from miracle_hip import hip as module
    b = HIPBackend()
    handle = b.empty((3, 5)).handle
    again = b.empty((15,))
    assert again.handle == handle and b._pooled == 0
    big = [b.empty((8 << 20,)) for _ in range(3)]     # 32 MiB each: two fit the pool
    del big
    assert b._pooled == module._POOL_BYTES
    np.testing.assert_array_equal(b.read(b.upload(np.arange(6, dtype=np.float32))), np.arange(6, dtype=np.float32))

    class Full:   # the library with its first allocation refused
        def __init__(self, lib):
            self.lib, self.asked = lib, 0

        def __getattr__(self, name):
            return getattr(self.lib, name)

        def mr_alloc(self, *args):
            self.asked += 1
            return 3 if self.asked == 1 else self.lib.mr_alloc(*args)

    b.lib = Full(b.lib)
    other = b.empty((7,))
    assert b.lib.asked == 2 and b._pooled == 0        # given back, then asked again
    b.lib.asked = 0
    with pytest.raises(HIPError, match="allocate"):
        b.empty((9,))
    del other
    b.close()
    assert b._pooled == 0


def test_full_pool_gives_up_its_oldest_sizes():
    """Sizes that do not come back fill the pool once; after that a new size is
    recycled all the same, the stale ones go first and the bound holds."""
    from miracle_hip import HIPBackend
    from miracle_hip import hip as module
    b = HIPBackend()
    for i in range(20):                       # 20 x 4 MiB and some: more than the pool
        del_me = b.empty(((1 << 20) + 64 * i,))
        del del_me
    assert module._POOL_BYTES - (5 << 20) < b._pooled <= module._POOL_BYTES
    first, last = 4 * (1 << 20), 4 * ((1 << 20) + 64 * 19)
    assert not b._pool.get(first) and len(b._pool[last]) == 1
    handle = b.empty((1000,)).handle
    assert b._pool[4000] == [handle]
    more = [b.empty((2 << 20,)) for _ in range(6)]
    del more
    assert b._pool[4000] == [handle] and len(b._pool[8 << 20]) == 6 and b._pooled <= module._POOL_BYTES
    assert b._pooled == sum(size * len(kept) for size, kept in b._pool.items())
    huge = b.empty((17 << 20,))               # past the pool's bytes: it displaces nothing
    pooled = b._pooled
    del huge
    assert b._pooled == pooled and b._pool[4000] == [handle]
    b.close()


def _free_bytes(b):
    import ctypes as C
    free, total = C.c_size_t(), C.c_size_t()
    assert b.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0   # of the runtime the library is linked to
    return free.value


def test_model_buffers_claim_cached_blocks():
    """A model's allocation that finds no memory takes back what the context
    only keeps: freed tensors of both pools and the operations' workspace."""
    from miracle_hip import HIPBackend
    bundle = presets.micro("flashnano-1.7")
    b = HIPBackend()
    x, w = b.upload(np.ones((4096, 2048), np.float32)), b.upload_weight(np.ones((2048, 2048), np.float16))
    b.read(b.linear(x, w))                    # its workspace: three planes of x, 48 MiB
    tensor = b.empty((1 << 28,))              # 1 GiB, past the pool: the library's free blocks
    del x, w, tensor
    free = _free_bytes(b)
    assert b.lib.mr_debug_fail_alloc(b.ctx) == 0
    with MiracleModel(ModelConfig.from_dict(bundle), synthetic.micro_weights(bundle), backend=b,
                      context_length=32) as model:
        assert not b._pool
        model.prefill([1, 2, 3])
        # a gibibyte of blocks and the workspace came back, less the model's own few buffers
        assert _free_bytes(b) > free + (1 << 30) + (16 << 20)
    y = b.read(b.linear(b.upload(np.ones((40, 128), np.float32)), b.upload_weight(np.ones((8, 128), np.float16))))
    np.testing.assert_array_equal(y, np.full((40, 8), 128, np.float32))
    b.close()


def test_workspace_is_one_block_as_large_as_needed():
    """Linears of growing and shrinking sizes leave one workspace, of the
    largest call's size, not one a size."""
    from miracle_hip import HIPBackend
    b = HIPBackend()
    w = b.upload_weight(np.ones((256, 2048), np.float16))
    xs = [b.upload(np.ones((rows, 2048), np.float32)) for rows in (8192, 700, 1400, 2600, 5100, 8192)]
    b.read(b.linear(xs[0], w))
    free = _free_bytes(b)
    for x in xs:
        np.testing.assert_array_equal(b.read(b.linear(x, w)), np.full((x.shape[0], 256), 2048, np.float32))
    # the outputs' own blocks: 1 MiB a thousand rows
    assert _free_bytes(b) > free - (32 << 20)
    b.close()
