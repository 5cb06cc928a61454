"""CPU-only tests of the pure-host pieces of libpegainfer_qwen3.so against the oracle / the
reference's own unit tests (pegainfer-core/src/page_pool.rs:124-199, kv_pool.rs:290-310,
batch_decode_buffers.rs)."""
import ctypes
import os

import numpy as np
import pytest

from oracle import ops as O
from pegainfer_amd import ffi


@pytest.fixture(scope="module")
def H(built_libs):
    return ffi.host_lib()


def test_host_library_exports_every_declared_symbol(built_libs):
    import subprocess
    out = subprocess.run(["nm", "-D", "--defined-only", built_libs[1]], stdout=subprocess.PIPE, text=True).stdout
    exported = {ln.split()[-1] for ln in out.splitlines() if ln.strip()}
    declared = []
    for header in ("pegainfer_qwen3.h", "pegainfer_qwen35.h", "pegainfer_scheduler.h", "pegainfer_comm.h"):
        declared += ffi.declared_symbols(header)
    assert "pegainfer_comm_all_reduce_bf16_via_f32" in declared and "pegainfer_ep_dispatch_send" in declared
    missing = sorted(set(declared) - exported)
    assert not missing, missing


def test_page_pool_order_and_all_or_nothing(H):
    pool = H.pegainfer_pagepool_create(6)
    try:
        buf = np.zeros(8, dtype=np.int32)
        assert H.pegainfer_pagepool_acquire(pool, 3, buf.ctypes.data) == 3
        assert buf[:3].tolist() == [0, 1, 2]                      # page_pool.rs:36: pops yield 0,1,2,...
        assert H.pegainfer_pagepool_available(pool) == 3
        assert H.pegainfer_pagepool_acquire(pool, 4, buf.ctypes.data) == -1   # all-or-nothing
        assert H.pegainfer_pagepool_available(pool) == 3
        rel = np.array([0, 1, 2], dtype=np.int32)
        H.pegainfer_pagepool_release(pool, rel.ctypes.data, 3)
        assert H.pegainfer_pagepool_available(pool) == 6
        assert H.pegainfer_pagepool_acquire(pool, 6, buf.ctypes.data) == 6
        assert buf[:6].tolist() == [0, 1, 2, 3, 4, 5]             # released pages come back in order
        assert H.pegainfer_pagepool_acquire(pool, 0, buf.ctypes.data) == 0
    finally:
        H.pegainfer_pagepool_destroy(pool)


def test_bucket_for(H):
    for bs in range(1, 65):
        assert H.pegainfer_bucket_for(bs) == O.bucket_for(bs)
    assert H.pegainfer_bucket_for(65) == -1


@pytest.mark.parametrize("lens,padded", [([1024], 1), ([20000, 5], 2), ([100], 1), ([1500, 40, 7, 3000], 4),
                                         ([4096] * 8, 8), ([1], 1)])
def test_reference_split_plan_matches_oracle(H, lens, padded):
    """policy 0 == BatchDecodeBuffers::sync_split_kv_meta + attention_path, bit for bit."""
    slots = padded * 64
    ri, kt = np.zeros(slots, np.int32), np.zeros(slots, np.int32)
    oi, va = np.zeros(padded + 1, np.int32), np.zeros(slots, np.uint8)
    chunk, use = np.zeros(1, np.int32), np.zeros(1, np.int32)
    L = np.asarray(lens, np.int32)
    n = H.pegainfer_split_kv_plan(0, len(lens), L.ctypes.data, padded, 8, ri.ctypes.data, kt.ctypes.data,
                                  oi.ctypes.data, va.ctypes.data, chunk.ctypes.data, use.ctypes.data)
    ref = O.split_kv_plan(lens, padded)
    assert n == ref["padded_slots"] and chunk[0] == ref["kv_chunk_size"]
    assert np.array_equal(ri, ref["request_indices"]) and np.array_equal(kt, ref["kv_tile_indices"])
    assert np.array_equal(oi, ref["o_indptr"]) and np.array_equal(va, ref["block_valid_mask"])
    assert bool(use[0]) == O.attention_path_is_split(padded, max(lens))


@pytest.mark.parametrize("lens,padded", [([1024], 1), ([10000], 1), ([100], 1), ([4096] * 8, 8), ([2000, 30], 2)])
def test_mi355x_split_policy_invariants(H, lens, padded):
    """policy 1 may pick any chunking, but must cover every token exactly once with <= 64 chunks."""
    slots = padded * 64
    ri, kt = np.zeros(slots, np.int32), np.zeros(slots, np.int32)
    oi, va = np.zeros(padded + 1, np.int32), np.zeros(slots, np.uint8)
    chunk, use = np.zeros(1, np.int32), np.zeros(1, np.int32)
    L = np.asarray(lens, np.int32)
    H.pegainfer_split_kv_plan(1, len(lens), L.ctypes.data, padded, 8, ri.ctypes.data, kt.ctypes.data,
                              oi.ctypes.data, va.ctypes.data, chunk.ctypes.data, use.ctypes.data)
    c = int(chunk[0])
    assert c % 16 == 0 and c >= 64
    for r, n in enumerate(lens):
        tiles = kt[oi[r]:oi[r + 1]]
        assert np.all(ri[oi[r]:oi[r + 1]] == r) and tiles.tolist() == list(range(len(tiles)))
        assert len(tiles) <= 64 and (len(tiles) - 1) * c < n <= len(tiles) * c
    assert va[:oi[len(lens)]].all() and not va[oi[len(lens)]:].any()


@pytest.mark.parametrize("lens,padded,chunk,chunks", [
    ([1024], 1, 64, [16]),            # 64-token chunks (the floor): unchanged by round 5
    ([2000], 1, 112, [18]),           # 2000 / 20 = 100 -> 112: one round of the 8 waves, 16-aligned as before
    ([4096], 1, 256, [16]),           # 4096 / 20 = 205 -> 208 -> whole rounds of 8 waves: 256
    ([10000], 1, 512, [20]),          # 10 000 / 20 = 500 -> 512: four balanced rounds (18 x 560 before)
    ([1030, 777], 2, 112, [10, 7]),   # two requests share the budget: 10 chunks each at most
    ([540, 300], 2, 64, [9, 5]),      # ... and below 10 x 64 tokens the chunks are the un-capped plan's 64
])
def test_mi355x_fused_form_plan_of_round_5(H, lens, padded, chunk, chunks):
    """the fused attention + o_proj plan (pegainfer_split_kv_plan's default): at most 20 chunks shared by <= 2 requests,
    chunks above 128 tokens rounded up to whole rounds of the 8-wave workgroup (profiles/r5_long_ctx_chunks_ab.txt)"""
    slots = padded * 64
    ri, kt = np.zeros(slots, np.int32), np.zeros(slots, np.int32)
    oi, va = np.zeros(padded + 1, np.int32), np.zeros(slots, np.uint8)
    c, use = np.zeros(1, np.int32), np.zeros(1, np.int32)
    L = np.asarray(lens, np.int32)
    n = H.pegainfer_split_kv_plan(1, len(lens), L.ctypes.data, padded, 8, ri.ctypes.data, kt.ctypes.data,
                                  oi.ctypes.data, va.ctypes.data, c.ctypes.data, use.ctypes.data)
    got = [int(oi[r + 1] - oi[r]) for r in range(len(lens))]
    assert int(c[0]) == chunk and got == chunks, (int(c[0]), got)
    assert sum(got) <= 20 and n == padded * (32 // padded) and use[0] == 1


def test_native_safetensors_reader_matches_python(tmp_path):
    """The C++ mmap reader (csrc/host/safetensors_loader.h: JSON header parser, single file / HF directory with
    model.safetensors.index.json shards) sees the same tensors, shapes, dtypes and bytes as a Python parse."""
    import ctypes
    import json
    import struct
    from pegainfer_amd import ffi
    lib = ffi.host_lib()
    golden = os.path.join(os.path.dirname(__file__), "golden")

    def py_parse(fp):
        with open(fp, "rb") as f:
            n = struct.unpack("<Q", f.read(8))[0]
            header = json.loads(f.read(n))
            blob = np.frombuffer(f.read(), dtype=np.uint8)
        return {k: (v["dtype"], v["shape"], blob[v["data_offsets"][0]:v["data_offsets"][1]])
                for k, v in header.items() if k != "__metadata__"}

    def probe(path, name):
        shape, ndim, dt = (ctypes.c_int64 * 4)(), ctypes.c_int32(), ctypes.create_string_buffer(8)
        bsum, nt = ctypes.c_uint64(), ctypes.c_int32()
        rc = lib.pegainfer_safetensors_probe(os.fsencode(path), name.encode(), ctypes.addressof(shape),
                                             ctypes.addressof(ndim), ctypes.addressof(dt), ctypes.addressof(bsum),
                                             ctypes.addressof(nt))
        return rc, list(shape[:ndim.value]), dt.value.decode(), bsum.value, nt.value

    def checksum(b):
        return int((b.astype(np.uint64) * (1 + (np.arange(b.size, dtype=np.uint64) & 0xFF))).sum(dtype=np.uint64))

    for fn in ("qwen3_tiny.safetensors", "qwen35_tiny.safetensors"):
        fp = os.path.join(golden, fn)
        ref = py_parse(fp)
        for name, (dtype, shape, data) in ref.items():
            rc, shp, dt, bs, nt = probe(fp, name)
            assert (rc, shp, dt, nt) == (0, shape, dtype, len(ref)) and bs == checksum(data), name
    assert probe(os.path.join(golden, "qwen3_tiny.safetensors"), "no.such.tensor")[0] == -2
    assert probe(str(tmp_path / "missing.safetensors"), "x")[0] == -1
    # sharded HF directory: two shard files + index
    ref = py_parse(os.path.join(golden, "qwen3_tiny.safetensors"))
    names = sorted(ref)
    d = tmp_path / "model"
    d.mkdir()
    weight_map = {}
    for si, part in enumerate((names[:5], names[5:])):
        header, blobs, off = {}, [], 0
        for nme in part:
            dtype, shape, data = ref[nme]
            header[nme] = {"dtype": dtype, "shape": shape, "data_offsets": [off, off + data.size]}
            blobs.append(data.tobytes())
            off += data.size
            weight_map[nme] = f"model-{si:05d}-of-00002.safetensors"
        hj = json.dumps(header, separators=(",", ":")).encode()
        with open(d / f"model-{si:05d}-of-00002.safetensors", "wb") as f:
            f.write(struct.pack("<Q", len(hj)) + hj + b"".join(blobs))
    (d / "model.safetensors.index.json").write_text(json.dumps({"metadata": {"total_size": 1}, "weight_map": weight_map}))
    for nme in (names[0], names[-1]):
        rc, shp, dt, bs, nt = probe(str(d), nme)
        assert (rc, shp, dt, nt) == (0, ref[nme][1], ref[nme][0], len(ref)) and bs == checksum(ref[nme][2])


@pytest.fixture(scope="module")
def tables(tmp_path_factory):
    """csrc/host/row_tiles.h behind C entries"""
    import subprocess
    d = tmp_path_factory.mktemp("tables")
    (d / "t.cpp").write_text('#include "row_tiles.h"\nextern "C" int wide_rows(const int32_t* lens, int n, int T, int per, int kv, int keys) '
                             '{ return ptiles::wide_rows(lens, n, T, per, kv, keys); }\n'
                             'extern "C" int flat(const int32_t* lens, const int32_t* begin, int n, int heads, int most, int32_t* table, int room) {\n'
                             '  const size_t tiles = ptiles::flat_count(lens, n, heads, most);\n'
                             '  if ((int)tiles <= room) ptiles::flat_cut(lens, n, heads, most, tiles, table, [&](int i) { return begin[i]; });\n'
                             '  return (int)tiles; }\n')
    host = os.path.join(os.path.dirname(os.path.abspath(ffi.__file__)), "csrc", "host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-I", host, "-o", str(d / "t.so"), str(d / "t.cpp")], check=True)
    return ctypes.CDLL(str(d / "t.so"))


@pytest.mark.parametrize("lens,heads,kv,keys,rows", [
    ([1024], 16, 4, 1024, 64), ([128], 16, 4, 128, 64), ([128], 16, 4, 16512, 64),      # 128 workgroups of 16 rows and more: their keys were not dealt
    ([64], 16, 4, 64, 32), ([64], 16, 4, 640, 32), ([64], 16, 4, 641, 16), ([64], 16, 4, 4160, 16), ([127], 16, 4, 640, 64), ([124], 16, 4, 641, 16),
    ([32], 16, 4, 32, 16),                                                               # too few workgroups of wide tiles
    ([64, 1, 1, 1], 16, 4, 4097, 16),                                                    # one long context among short ones
    ([1] * 8, 64, 4, None, 16), ([1] * 31, 64, 4, None, 16), ([1] * 32, 64, 4, None, 32), ([1] * 64, 128, 4, None, 64), ([1] * 64, 16, 4, None, 16),
    ([1024], 16, 0, 1024, 16)])
def test_wide_attention_tiles_leave_no_key_split_behind(tables, lens, heads, kv, keys, rows):
    """short of 128 workgroups the 16-row tiles deal a long context's keys to up to 512, so wide tiles are for short ones; decoding steps
    (keys None: the choice may not depend on the contexts) take them only where nothing was dealt"""
    a = np.array(lens, np.int32)
    assert tables.wide_rows(ctypes.c_void_p(a.ctypes.data), len(lens), int(a.sum()), heads // max(kv, 1), kv, 2 ** 31 - 1 if keys is None else keys) == rows


@pytest.mark.parametrize("lens,begin,heads", [([3], [0], 8), ([1, 1], [70, 5], 16), ([900, 0, 301, 64], [0, 9, 700, 0], 16), ([1] * 100, list(range(0, 6400, 64)), 3),
                                              ([33, 1000], [5000, 0], 7)])
def test_latent_attention_tiles_hold_every_row_once_the_longest_first(tables, lens, begin, heads):
    a, b, t = np.array(lens, np.int32), np.array(begin, np.int32), np.full(20000, -1, np.int32)
    n = tables.flat(*(ctypes.c_void_p(x.ctypes.data) for x in (a, b)), len(lens), heads, 64, ctypes.c_void_p(t.ctypes.data), 10000)
    row0, rows = t[:n], t[n:2 * n]
    entry, pos = np.repeat(np.arange(len(lens)), a), np.concatenate([np.arange(s, s + k) for s, k in zip(begin, lens)])
    order = np.argsort(row0, kind="stable")
    assert n and (rows > 0).all() and (rows <= 64).all() and (t[2 * n:] == -1).all()
    assert (row0[order] + rows[order] == np.append(row0[order][1:], a.sum() * heads)).all() and row0.min() == 0
    first, last = row0 // heads, (row0 + rows - 1) // heads
    assert (entry[first] == entry[last]).all()
    steps = pos[last] // 64
    assert (np.diff(steps) <= 0).all() if n >= 64 else (order == np.arange(n)).all()


def test_optional_scratch_is_given_up_when_there_is_no_memory(tmp_path):
    """csrc/host/optional_scratch.h with an allocator that refuses more than 1000 bytes: a refusal leaves nothing behind, smaller needs are met
    afterwards, everything is released once"""
    import subprocess
    (tmp_path / "t.cpp").write_text(r"""
#include <cstdlib>
#include <set>
#include "optional_scratch.h"
int main() {
  std::set<void*> live;
  pq::OptionalScratch s;
  auto alloc = [&](size_t n) -> void* { if (n > 1000) return nullptr; void* p = std::malloc(n); live.insert(p); return p; };
  auto release = [&](float* p) { if (!live.erase(p)) std::exit(9); std::free(p); };
  if (!s.grow(0, alloc, release) || s.p) return 1;
  if (!s.grow(100, alloc, release) || !s.p || s.cap != 100) return 2;
  float* first = s.p;
  if (!s.grow(60, alloc, release) || s.p != first || s.cap != 100) return 3;
  if (s.grow(251, alloc, release) || s.p || s.cap || !live.empty()) return 4;
  if (!s.grow(0, alloc, release) || s.p) return 5;
  if (!s.grow(250, alloc, release) || !s.p || s.cap != 250 || live.size() != 1) return 6;
  s.drop(release);
  s.drop(release);
  return s.p || s.cap || !live.empty() ? 7 : 0;
}
""")
    host = os.path.join(os.path.dirname(os.path.abspath(ffi.__file__)), "csrc", "host")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", host, "-o", str(tmp_path / "t"), str(tmp_path / "t.cpp")], check=True)
    assert subprocess.run([str(tmp_path / "t")]).returncode == 0


def test_a_capture_that_fails_leaves_no_graph_behind(tmp_path):
    """csrc/host/graph_capture.h over a runtime of counters: the recording is destroyed once whether a launch was refused, the capture or the instantiation
    failed or all went well, and only then is there an executable graph"""
    import subprocess
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(r"""
#pragma once
enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999 };
typedef int* hipStream_t;
typedef int* hipGraph_t;
typedef int* hipGraphExec_t;
inline int graphs = 0, execs = 0, dummy = 0;
inline bool bad_end = false, bad_make = false;
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { if (bad_end) return hipErrorUnknown; ++graphs; *g = &dummy; return hipSuccess; }
inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, void*, char*, unsigned long) {
  *e = &dummy;
  if (bad_make) return hipErrorUnknown;
  ++execs;
  return hipSuccess;
}
inline hipError_t hipGraphDestroy(hipGraph_t) { --graphs; return hipSuccess; }
""")
    (tmp_path / "t.cpp").write_text(r"""
#include "graph_capture.h"
int main() {
  hipGraphExec_t e = &dummy;
  if (pst::end_capture(nullptr, false, &e) != hipSuccess || e || graphs || execs) return 1;      // a launch was refused
  bad_end = true;
  if (pst::end_capture(nullptr, true, &e) == hipSuccess || e || graphs || execs) return 2;
  bad_end = false; bad_make = true;
  if (pst::end_capture(nullptr, true, &e) == hipSuccess || e || graphs || execs) return 3;
  bad_make = false;
  return pst::end_capture(nullptr, true, &e) != hipSuccess || !e || graphs || execs != 1 ? 4 : 0;
}
""")
    host = os.path.join(os.path.dirname(os.path.abspath(ffi.__file__)), "csrc", "host")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(tmp_path), "-I", host, "-o", str(tmp_path / "t"), str(tmp_path / "t.cpp")], check=True)
    assert subprocess.run([str(tmp_path / "t")]).returncode == 0
    sources = [os.path.join(host, f) for f in os.listdir(host) if f.endswith((".cpp", ".h")) and f != "graph_capture.h"]
    assert not [f for f in sources if "hipStreamEndCapture" in open(f).read()]      # every runtime ends its captures here


def test_the_graph_that_goes_is_the_one_not_asked_for_the_longest(tmp_path):
    """csrc/host/graph_cache.h: what was asked for stays beyond what was added earlier, one goes per addition, everything is destroyed once"""
    import subprocess
    (tmp_path / "t.cpp").write_text(r"""
#include <set>
#include "graph_cache.h"
int main() {
  int things[16];
  std::multiset<int*> gone;
  auto destroy = [&](int* p) { gone.insert(p); };
  pst::GraphCache<int, int*> c(3);
  if (c.find(0)) return 1;
  for (int k = 0; k < 3; ++k) c.add(k, things + k, destroy);
  if (!gone.empty() || c.find(0) != things || c.find(2) != things + 2) return 2;
  c.add(3, things + 3, destroy);                              // 1 goes
  if (gone != std::multiset<int*>{things + 1} || c.find(1) || c.find(0) != things) return 3;
  c.add(4, things + 4, destroy);                              // 2 goes
  if (gone != std::multiset<int*>{things + 1, things + 2} || c.find(2) || c.find(3) != things + 3 || c.find(0) != things || c.find(4) != things + 4) return 4;
  c.drop(destroy);
  if (gone != std::multiset<int*>{things, things + 1, things + 2, things + 3, things + 4} || c.find(0) || c.find(4)) return 5;
  c.add(0, things + 5, destroy);
  return c.find(0) != things + 5 || gone.size() != 5 ? 6 : 0;
}
""")
    host = os.path.join(os.path.dirname(os.path.abspath(ffi.__file__)), "csrc", "host")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", host, "-o", str(tmp_path / "t"), str(tmp_path / "t.cpp")], check=True)
    assert subprocess.run([str(tmp_path / "t")]).returncode == 0


def test_scratch_of_the_chunk_forms_is_bounded(built_libs):
    """256 MB of states (or one chunk's) however long the step, and the gates' 768 bytes per chunk and head beside them"""
    L = ffi.lib()
    for heads, dim, vdim in ((32, 128, 64), (1, 5, 33), (64, 256, 1024)):
        per = L.pegainfer_ssd_scan_workspace(1, heads, dim, vdim)
        assert L.pegainfer_ssd_scan_workspace(2, heads, dim, vdim) == 2 * per and L.pegainfer_ssd_scan_workspace(0, heads, dim, vdim) == 0
        for n in (16, 1000, 30000):
            assert L.pegainfer_ssd_scan_workspace(n, heads, dim, vdim) == min(n, max(1, 2 ** 26 // per)) * per
            mem = L.pegainfer_gated_matrix_memory_workspace(n, heads, dim, vdim) - n * heads * 192
            assert 0 < mem <= max(2 ** 26, L.pegainfer_gated_matrix_memory_workspace(1, heads, dim, vdim))
