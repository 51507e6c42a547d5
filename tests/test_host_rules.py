"""The host side of the library without a device: which kernels a call
launches, with which grids, and which calls it refuses.  A child process loads
tests/hip_stub.cpp (a recording stand-in for the HIP runtime) before liblgx.so
and runs the calls on made-up pointers."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PTR = 1 << 41                     # any non-NULL device address: nothing runs

CHILD = r"""
import ctypes as C, json, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
stub.stub_log.restype = C.c_char_p
import logicaffeine_amd as lgx
L = lgx.lib()
h = C.c_void_p()
lgx._check(L.lgx_ctx_create(0, b"stub", C.byref(h)))
P = 1 << 41
for line in sys.stdin:
    name, args = json.loads(line)
    def arg(a):
        if isinstance(a, dict):
            return C.byref(lgx.Q8MatrixC(P, P, a["n"], a["k"], lgx.Q8_T16))
        if isinstance(a, list) and a and isinstance(a[0], dict):
            return (lgx.Q8MatrixC * len(a))(*[lgx.Q8MatrixC(P, P, w["n"], w["k"], lgx.Q8_T16) for w in a])
        if isinstance(a, list):
            return (C.c_void_p * len(a))(*a)
        return a
    stub.stub_reset()
    st = getattr(L, name)(h, *[arg(a) for a in args])
    print(json.dumps([lgx.STATUS_NAMES.get(st, st), stub.stub_log().decode().splitlines()]), flush=True)
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    """calls -> [(status, [kernel launches as (name, gx, gy, gz, block)], bytes allocated)]"""
    so = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-fPIC", "-shared", "-std=c++17", f"-I{rocm}/include", "-o", so,
                    os.path.join(ROOT, "tests", "hip_stub.cpp")], check=True)

    def run(calls, **env):
        r = subprocess.run([sys.executable, "-c", CHILD, so], cwd=ROOT, text=True, capture_output=True, timeout=300,
                           input="".join(json.dumps(c) + "\n" for c in calls), env={**os.environ, **env})
        assert r.returncode == 0, r.stderr[-4000:]
        out = []
        for line in r.stdout.splitlines():
            st, log = json.loads(line)
            words = [ln.split() for ln in log]
            out.append((st, [(w[0], *map(int, w[1:])) for w in words if w[0] != "malloc"],
                        sum(int(w[1]) for w in words if w[0] == "malloc")))
        assert len(out) == len(calls)
        return out

    return run


def gemm(name, n, k, m):
    return [name, [dict(n=n, k=k), PTR, PTR, m, PTR, None]]


def least_scratch(n, k, m):
    """T16 copy of the rows and the partials of range groups of 4, the least
    that a product of 33 and more rows can do with."""
    ng = -(-k // 4096)
    return -(-m // 16) * 16 * k + (ng * m * n * 4 if ng > 1 else 0)


@pytest.mark.parametrize("n,k", [(6400, 18944), (4032, 32768), (3584, 18944), (37888, 3584), (896, 4864),
                                 (1536, 8960), (16, 32768), (8192, 4160)])
def test_noalloc_takes_every_product_whose_least_scratch_fits(host, n, k):
    """The row tile and the range groups chosen for speed must not cost a
    product its place in the fixed scratch (6400 x 18944 at 122..127 rows and
    4032 x 32768 at 114..127 fit only with groups of 4)."""
    ms = list(range(33, 161)) + list(range(161, 2049, 37))
    for m, (st, launches, alloc) in zip(ms, host([gemm("lgx_q8_gemm_noalloc", n, k, m) for m in ms])):
        fits = least_scratch(n, k, m) <= 32 << 20
        assert st == ("LGX_OK" if fits else "LGX_OUT_OF_BOUNDS"), (m, st)
        assert alloc == 0 and bool(launches) == fits


def prefill(B, P, hq, hkv, d, max_seq):
    return ["lgx_gqa_prefill_attn", [PTR] * 5 + [B, P, hq, hkv, d, -(-max_seq // 16), 1000, max_seq, PTR, None]]


@pytest.mark.parametrize("B,P,hq,hkv,d,max_seq", [
    (4096, 1, 8, 8, 64, 129 * 256),       # 4.2 million (sequence, KV head, chunk) triples
    (65535, 4, 8, 1, 128, 100 * 256),
    (1, 1, 1, 1, 64, 1 << 29),            # 2 million chunks
    (8192, 17, 64, 8, 64, 2048),          # a run and a quarter of query blocks
    (1, 3, 7, 1, 128, 65537 * 256), (3, 3, 12, 2, 128, 32769 * 256),  # more chunks than a grid's y
    (16, 2, 28, 4, 128, 2000), (3, 33, 12, 2, 64, 100)])
def test_prefill_attention_launches_every_block(host, B, P, hq, hkv, d, max_seq):
    """Every (sequence, KV head, block of 32 / heads or 16 / heads rows, chunk) has a
    workgroup, the blocks along x in whole eights, several chunks to an eight
    where a chunk has up to four; at most 8 / 5 and 7 runs more than are needed."""
    (st, launches, _), = host([prefill(B, P, hq, hkv, d, max_seq)])
    assert st == "LGX_OK"
    name, gx, gy, gz, block = launches[0]
    rows = 16 if name.startswith("lgx_k_attn_prefill16") else 32
    assert name == f"lgx_k_attn_prefill{'16' if rows == 16 else ''}_d{d}_g{hq // hkv}" and block == 256
    nqb, ncg = -(-P // (rows // (hq // hkv))), -(-max_seq // 256)
    need = B * hkv * nqb
    assert gx % 8 == 0
    runs = need // nqb * -(-nqb // 4)
    fold = 8 // runs if runs <= 4 else 1
    assert need * fold <= gx <= need * fold * 8 / 5 + 8 * 4
    assert ncg <= gy * gz * fold < ncg + gy * fold + fold


@pytest.mark.parametrize("n,k,m", [(16448, 64, 4194240), (16448, 64, 4194240 - 63), (128, 64, 4194240)])
def test_products_of_the_most_rows_are_launched_whole(host, n, k, m):
    """Products past the 2^32 threads of one launch go in several, alone and
    in a group, and their workgroups cover every 64 x 64 tile."""
    calls = [gemm("lgx_q8_gemm", n, k, m),
             ["lgx_q8_gemm_quantize_group", [1, [dict(n=n, k=k)], [PTR], m, [PTR], None]]]
    for st, launches, _ in host(calls):
        assert st == "LGX_OK"
        tiles = sum(gx for name, gx, *_ in launches if "gemm_tiled64" in name)
        assert -(-n // 64) * -(-m // 64) <= tiles < -(-n // 64) * (-(-m // 64) + 2) + 16


@pytest.mark.parametrize("n,k", [(37888, 3584), (151936, 896), (3584, 18944), (512, 32768)])
def test_rows_65_to_96_are_not_padded_to_128(host, n, k):
    """Three 32-row tiles of a product, not two of 64 with the last half empty."""
    for m, (st, launches, _) in zip(range(65, 97), host([gemm("lgx_q8_gemm", n, k, m) for m in range(65, 97)])):
        names = [name for name, *_ in launches if "gemm_tiled" in name]
        assert st == "LGX_OK" and len(names) == 1 and names[0].startswith("lgx_k_q8_gemm_tiled32"), (m, names)


@pytest.mark.parametrize("shapes,ms,rows", [
    ([(37888, 3584)], range(97, 256, 6), 64), ([(37888, 3584)], range(17, 97, 5), 32),
    ([(18944, 3584)] * 2 + [(3584, 18944)], range(97, 300, 9), 64), ([(8960, 1536)] * 2, range(97, 193, 9), 32),
    ([(4864, 896), (896, 4864)], [100, 160, 255], 32), ([(8960, 1536)], [257, 520], 64)])
def test_grouped_products_take_the_row_tile_of_their_whole_grid(host, shapes, ms, rows):
    """One rule for a product in one group and for several matrices in one
    launch (37888 x 3584 alone and grouped took different tiles at 97..255
    rows)."""
    def group(m):
        return ["lgx_q8_gemm_quantize_group", [len(shapes), [dict(n=n, k=k) for n, k in shapes], [PTR] * len(shapes), m,
                                               [PTR] * len(shapes), None]]
    for m, (st, launches, _) in zip(ms, host([group(m) for m in ms])):
        names = [name for name, *_ in launches if "gemm_tiled" in name]
        assert st == "LGX_OK" and names == [f"lgx_k_q8_gemm_tiled{rows}_group"], (m, names)
