"""CPU: libcoopt_amd.so loads, binds torch's HIP runtime, exports every symbol of
include/coopt_amd.h, and rejects bad arguments with an error code + message before any launch.
No kernel is launched here."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch  # noqa: F401  (must precede the library load)

from iitj_llm_coopt_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "coopt_amd.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(coopt_\w+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def test_every_declared_symbol_is_exported_and_bound(lib):
    names = declared_functions()
    assert len(names) >= 10
    for name in names:
        assert hasattr(lib, name), name
        assert name in _lib.SIGNATURES, f"{name} has no ctypes signature"
    assert set(_lib.SIGNATURES) == set(names)


def test_single_hip_runtime_is_mapped(lib):
    hip = _lib._hip_libs_mapped()
    assert len(hip) == 1 and "torch" in hip[0], hip


def test_runtime_version_matches_torch(lib):
    v = _lib.runtime_version()
    major, minor = v // 10000000, (v // 100000) % 100
    assert f"{major}.{minor}" == ".".join(torch.version.hip.split(".")[:2]), (v, torch.version.hip)


def test_workspace_sizes_are_positive_and_monotone(lib):
    a = lib.coopt_verify_attention_workspace(32, 32, 8, 128, 5, 4101)
    b = lib.coopt_verify_attention_workspace(64, 32, 8, 128, 9, 16393)
    assert 0 < a < b
    assert lib.coopt_verify_attention_workspace(0, 32, 8, 128, 5, 100) == 0
    c = lib.coopt_accept_sample_workspace(8, 4, 128256)
    d = lib.coopt_accept_sample_workspace(32, 4, 128256)
    assert 0 < c < d


def test_workspace_bytes_follow_the_sizes_values(lib):
    """Sizes given as 0-d arrays and tensors count by their value at the call, also when the same
    object holds another one later; what has no integer value is refused."""
    from iitj_llm_coopt_amd.attention import workspace_bytes

    small, large = workspace_bytes(2, 32, 8, 128, 5, 600), workspace_bytes(2, 32, 8, 128, 5, 6000)
    assert 0 < small < large
    keys = torch.tensor(600)
    assert workspace_bytes(2, 32, 8, 128, 5, keys) == small
    keys.fill_(6000)
    assert workspace_bytes(2, 32, 8, 128, 5, keys) == large
    assert workspace_bytes(2, 32, 8, 128, np.array(5), np.int64(6000)) == large
    assert workspace_bytes(batch=2, num_heads=32, num_kv_heads=8, head_dim=128, max_seqlen_q=5,
                           max_seqlen_k=600) == small
    for bad in (600.0, "600", None):
        with pytest.raises(TypeError):
            workspace_bytes(2, 32, 8, 128, 5, bad)


def _err(rc):
    assert rc == _lib.COOPT_EINVAL, rc
    msg = _lib.last_error()
    assert msg
    return msg


def test_kv_write_rejects_bad_arguments(lib):
    msg = _err(lib.coopt_kv_write(99, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 8,
                                  128, 16, 16, None))
    assert "cache_dtype" in msg
    assert "D must be" in _err(lib.coopt_kv_write(_lib.DT_BF16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
                                                  0, 0, 0, 0, 0, 0, 1, 8, 96, 16, 16, None))
    assert "null" in _err(lib.coopt_kv_write(_lib.DT_BF16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
                                             0, 0, 0, 0, 1, 8, 128, 16, 16, None))
    # misaligned k/v rows (pointer not 16-byte aligned): rejected before launch
    assert "aligned" in _err(lib.coopt_kv_write(_lib.DT_BF16, 8, 8, 1024, 128, 1024, 128, 16, 16,
                                                0, 0, 0, 0, 0, 0, 0, 0, 16, 1, 8, 128, 16, 16,
                                                None))
    # T == 0 is a no-op
    assert lib.coopt_kv_write(_lib.DT_BF16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
                              8, 128, 16, 16, None) == 0


def test_verify_attention_rejects_unsupported_shapes(lib):
    args = dict(kv=_lib.DT_BF16, B=2, Hq=32, Hkv=8, D=128, bs=16, mq=5, mk=100, bt=16)

    def call(**kw):
        a = {**args, **kw}
        return lib.coopt_verify_attention(a["kv"], 16, 4096, 128, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0,
                                          16, a["bt"], 16, 16, a["B"], a["Hq"], a["Hkv"], a["D"],
                                          a["bs"], 64, a["mq"], a["mk"], 0.088, 16, 4096, 128, 16,
                                          1 << 30, None)
    assert "head_dim" in _err(call(D=96))
    assert "multiple of Hkv" in _err(call(Hq=30))
    assert "<= 64" in _err(call(Hq=130, Hkv=2))   # more query heads per KV head than rows
    assert "power of two" in _err(call(bs=24))
    assert ">= 16" in _err(call(bs=8))
    assert "narrower" in _err(call(bt=3))
    assert "kv_dtype" in _err(call(kv=7))
    # INT8 without scales
    assert "scale" in _err(call(kv=_lib.DT_I8))


def test_verify_attention_reports_small_workspace(lib):
    rc = lib.coopt_verify_attention(_lib.DT_BF16, 16, 4096, 128, 16, 16, 0, 0, 0, 0, 0, 0, 0, 0,
                                    16, 16, 16, 16, 2, 32, 8, 128, 16, 64, 5, 100, 0.088, 16,
                                    4096, 128, 16, 8, None)
    assert rc == _lib.COOPT_EWORKSPACE and "workspace" in _lib.last_error()


# Windowed attention calls and the us they take in query windows of 64 and of 128 rows (MI355X, head
# dim 128, the longest context max_k): INT8?, B, Hq, Hkv, max_q, max_k, query rows.
WINDOWED = [
    (0, 1, 32, 8, 512, 512, 512, 14.8, 21.1), (0, 1, 32, 8, 512, 4096, 512, 65.1, 119.5),
    (0, 1, 32, 8, 512, 16384, 512, 240.6, 438.4), (1, 1, 32, 8, 512, 16384, 512, 321.4, 530.6),
    (0, 1, 32, 8, 2048, 4096, 2048, 197.4, 142.7), (1, 1, 32, 8, 2048, 16384, 2048, 1163.8, 740.5),
    (0, 5, 32, 8, 256, 4096, 276, 68.7, 120.6), (0, 17, 32, 8, 33, 4096, 113, 67.4, 121.5),
    (0, 17, 32, 8, 64, 4096, 144, 182.0, 123.8), (0, 17, 32, 8, 512, 16384, 592, 712.9, 448.8),
    (0, 32, 32, 8, 33, 4096, 188, 130.7, 166.8), (0, 32, 32, 8, 512, 1000, 667, 105.7, 31.8),
    (0, 4, 32, 8, 17, 4096, 68, 64.3, 119.9), (0, 4, 32, 8, 512, 4096, 2048, 240.2, 166.2),
    (0, 16, 32, 8, 128, 4096, 2048, 255.1, 177.6), (0, 40, 32, 8, 256, 256, 10240, 172.9, 75.7),
    (1, 40, 32, 8, 128, 4096, 5120, 862.0, 506.0),
    (0, 33, 32, 4, 1553, 1553, 1681, 114.1, 58.2), (0, 6, 32, 4, 107, 3996, 244, 63.5, 118.6),
]


def test_window_rows_are_the_faster_ones(lib):
    for int8, B, Hq, Hkv, max_q, max_k, rows, t64, t128 in WINDOWED:
        got = lib.coopt_verify_attention_window_rows(_lib.DT_I8 if int8 else _lib.DT_BF16, B, Hq, Hkv, 128,
                                                     max_q, max_k, rows)
        assert got == (128 if t128 < t64 else 64), (int8, B, Hq, Hkv, max_q, max_k, rows)
    # not windowed; refused shapes; rows unknown or short count as one a sequence
    q = lib.coopt_verify_attention_window_rows
    assert q(_lib.DT_BF16, 4, 32, 8, 128, 16, 4096, 64) == 0 and q(_lib.DT_BF16, 4, 32, 8, 128, 17, 4096, 68) == 64
    assert q(_lib.DT_BF16, 4, 130, 2, 128, 17, 4096, 68) == 0 and q(_lib.DT_BF16, 0, 32, 8, 128, 17, 4096, 0) == 0
    for B, max_q in ((1, 512), (16, 128), (70, 20)):
        assert q(_lib.DT_BF16, B, 32, 8, 64, max_q, 4096, 0) == q(_lib.DT_BF16, B, 32, 8, 64, max_q, 4096, max_q + B - 1)


def test_accept_sample_rejects_bad_arguments(lib):
    assert "logits_dtype" in _err(lib.coopt_accept_sample(5, 16, 100, 0, 0, 16, 100, 0, 16, 0,
                                                          16, 16, 1.0, 2, 4, 100, 16, 16, 0, 16,
                                                          1 << 20, None))
    assert "null" in _err(lib.coopt_accept_sample(_lib.DT_F32, 0, 100, 0, 0, 16, 100, 0, 16, 0,
                                                  16, 16, 1.0, 2, 4, 100, 16, 16, 0, 16, 1 << 20,
                                                  None))
    assert "stride" in _err(lib.coopt_accept_sample(_lib.DT_F32, 16, 50, 0, 0, 16, 100, 0, 16, 0,
                                                    16, 16, 1.0, 2, 4, 100, 16, 16, 0, 16,
                                                    1 << 20, None))
    rc = lib.coopt_accept_sample(_lib.DT_F32, 16, 100, 0, 0, 16, 100, 0, 16, 0, 16, 16, 1.0, 2, 4,
                                 100, 16, 16, 0, 16, 8, None)
    assert rc == _lib.COOPT_EWORKSPACE


def test_codec_rejects_bad_arguments(lib):
    assert "bits" in _err(lib.coopt_quantize(6, _lib.DT_BF16, 16, 4, 128, 16, 16, None))
    assert "even" in _err(lib.coopt_quantize(8, _lib.DT_BF16, 16, 4, 127, 16, 16, None))
    assert "out_dtype" in _err(lib.coopt_dequantize(8, 16, 16, 4, 128, _lib.DT_I8, 16, None))


def test_python_wrappers_refuse_cpu_tensors():
    import iitj_llm_coopt_amd as M

    x = torch.zeros(4, 128, dtype=torch.bfloat16)
    with pytest.raises(_lib.CooptError, match="no CPU fallback"):
        M.quantize(x, 8)
    with pytest.raises(_lib.CooptError, match="no CPU fallback"):
        M.sample(torch.zeros(2, 10), 1.0)


def test_accept_noalloc_rejects_sizes_beyond_its_scratch(lib):
    """The static-scratch accept entry point checks its size before touching the device."""
    cap = lib.coopt_accept_sample_noalloc_max_bytes()
    assert cap == 2 << 20
    assert lib.coopt_accept_sample_workspace(512, 8, 128256) <= cap
    need = lib.coopt_accept_sample_workspace(4096, 8, 262144)
    assert need > cap
    rc = lib.coopt_accept_sample_noalloc(_lib.DT_F32, 16, 262144, None, 0, 16, 262144, None, 16,
                                         None, 16, 16, 1.0, 4096, 8, 262144, 16, 16, 16, None)
    assert rc == _lib.COOPT_EWORKSPACE
    msg = _lib.last_error()
    assert "scratch" in msg and str(need) in msg and str(cap) in msg, msg
    assert lib.coopt_accept_sample_noalloc(_lib.DT_F32, 0, 1, None, 0, 0, 1, None, 0, None, 0, 0,
                                           1.0, 0, 4, 100, 0, 0, 0, None) == _lib.COOPT_OK
