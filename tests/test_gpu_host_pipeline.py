"""The host entry points copy through two pinned bounce buffers, chunk by
chunk, overlapping the host copies with the DMA.  With small odd chunk sizes
(PETJSON_XFER_CHUNK, read when a context first copies) every copy crosses
many chunk boundaries: pj_encode_host's output equals pj_encode_device's,
and pj_decode_host's / pj_decode_array_host's columns equal the device
decode's, byte for byte, on records of every configuration."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = r"""
import sys
import numpy as np, torch
import petjson as pj
codec = pj.Codec(0)
for cfg, n in ((1, 20000), (3, 30000), (5, 3000)):
    cols = pj.generate(cfg, n)
    dev = cols.to_device()
    for fmt in (pj.FORMAT_ARRAY, pj.FORMAT_NDJSON):
        want = codec.encode(dev, fmt).cpu().numpy().tobytes()
        got = codec.encode_host(cols, fmt)
        assert got == want, (cfg, fmt, len(got), len(want))
        d = torch.from_numpy(np.frombuffer(want, np.uint8).copy()).cuda()
        ref = codec.decode(d, array=fmt == pj.FORMAT_ARRAY)[0].to_host()
        host = (codec.decode_array_host if fmt == pj.FORMAT_ARRAY else codec.decode_host)(want)[0]
        for k in pj.COLS:
            assert np.array_equal(host[k], ref[k]), (cfg, fmt, k)
codec.close()
print("host pipeline ok")
"""


@pytest.mark.parametrize("chunk", [4099, 65537, 1 << 20])
def test_host_entry_points_across_chunks(chunk):
    env = dict(os.environ, PETJSON_XFER_CHUNK=str(chunk),
               PYTHONPATH=os.pathsep.join([os.path.join(ROOT, "micronaut3-bug_amd"), os.path.join(ROOT, "tests")]))
    r = subprocess.run([sys.executable, "-c", SCRIPT], capture_output=True, text=True, env=env, timeout=240)
    assert r.returncode == 0 and "host pipeline ok" in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]


STREAM = r"""
import numpy as np, torch
import petjson as pj
codec = pj.Codec(0)
parts = []
for cfg, n in ((3, 40000), (5, 4000)):
    buf = codec.encode(pj.generate(cfg, n).to_device(), pj.FORMAT_NDJSON).cpu().numpy().copy()
    pj.corrupt_ndjson(buf, 11 + cfg, 0.01)
    parts.append(buf.tobytes())
long_line = b'{"id":1,"name":"' + b"L" * 3_000_000 + b'","photoUrls":["u"],"tags":[]}\n'
data = parts[0] + b"\n\n" + long_line + parts[1] + b'{"name":"last","photoUrls":[]}'   # no final newline
d = torch.from_numpy(np.frombuffer(data, np.uint8).copy()).cuda()
ref, el_r, ec_r, res_r = codec.decode(d)
ref = ref.to_host()
el_r, ec_r = el_r.cpu().numpy(), ec_r.cpu().numpy()
host, el, ec, res = codec.decode_host(data)
for k in ("n_lines", "n_pets", "n_errors", "name_bytes", "cat_name_bytes", "n_urls", "url_bytes", "n_tags", "tag_name_bytes"):
    assert getattr(res, k) == getattr(res_r, k), (k, getattr(res, k), getattr(res_r, k))
for k in pj.COLS:
    assert np.array_equal(host[k], ref[k]), k
assert np.array_equal(el, el_r) and np.array_equal(ec, ec_r)
# capacities one short: PJ_ERR_CAPACITY, with the sizes the whole input needs
caps = pj.decode_bounds(len(data))
caps["cap_url_bytes"] = int(res_r.url_bytes) - 1
try:
    codec.decode_host(data, caps=caps)
    raise SystemExit("expected a capacity error")
except pj.PetJsonError as e:
    assert e.status == pj.PJ_ERR_CAPACITY, e
codec.close()
print("streamed decode ok")
"""


@pytest.mark.parametrize("segment,chunk", [(1_000_003, None), (4_194_301, 65537)])
def test_host_decode_streamed_in_segments(segment, chunk):
    """Inputs over PETJSON_DECODE_SEGMENT bytes (default: inputs over 512
    MiB, in 256 MiB segments) are decoded in segments cut after a newline,
    in a pipeline: the next segment copied in and the previous one's columns
    copied out while one decodes.  Columns, error lines and codes, and totals
    equal the one-shot device decode.  The input holds blank lines, 1%
    corrupted lines, a 3 MB line longer than a segment, skewed records, and a
    last line without its newline; capacities one short report
    PJ_ERR_CAPACITY.  With small bounce chunks (PETJSON_XFER_CHUNK) both copy
    directions cross many chunk boundaries while running at once."""
    env = dict(os.environ, PETJSON_DECODE_SEGMENT=str(segment),
               PYTHONPATH=os.pathsep.join([os.path.join(ROOT, "micronaut3-bug_amd"), os.path.join(ROOT, "tests")]))
    if chunk:
        env["PETJSON_XFER_CHUNK"] = str(chunk)
    r = subprocess.run([sys.executable, "-c", STREAM], capture_output=True, text=True, env=env, timeout=240)
    assert r.returncode == 0 and "streamed decode ok" in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]


PINNED = r"""
import ctypes as C
import numpy as np, torch
import petjson as pj
codec = pj.Codec(0)
buf = codec.encode(pj.generate(3, 60000).to_device(), pj.FORMAT_NDJSON).cpu().numpy().copy()
lines, codes = pj.corrupt_ndjson(buf, 7, 0.01)
ref, el_r, ec_r, res_r = codec.decode(torch.from_numpy(buf).cuda())
ref = ref.to_host()
n = buf.size
inp = pj.host_array(n, np.uint8)
inp[:] = buf
caps = pj.decode_bounds(n)
cp, cu, ct = caps["cap_pets"], caps["cap_urls"], caps["cap_tags"]
sizes = {"id": cp, "flags": cp, "status": cp, "name_off": cp + 1, "name_bytes": caps["cap_name_bytes"],
         "cat_id": cp, "cat_flags": cp, "cat_name_off": cp + 1, "cat_name_bytes": caps["cap_cat_name_bytes"],
         "photo_off": cp + 1, "url_off": cu + 1, "url_bytes": caps["cap_url_bytes"], "tag_off": cp + 1,
         "tag_id": ct, "tag_flags": ct, "tag_name_off": ct + 1, "tag_name_bytes": caps["cap_tag_name_bytes"]}
cols = pj.Columns(0, {k: pj.host_array(v, pj.DTYPES[k]) for k, v in sizes.items()}, dict(caps))
el, ec = pj.host_array(4096, np.uint64), pj.host_array(4096, np.uint8)
s = cols.struct()
res = pj.DecodeResult()
rc = codec.L.pj_decode_host(codec.ctx, C.c_void_p(inp.ctypes.data), n, C.byref(s), C.c_void_p(el.ctypes.data),
                            C.c_void_p(ec.ctypes.data), 4096, C.byref(res))
assert rc == 0, rc
assert res.n_pets == res_r.n_pets and res.n_errors == res_r.n_errors == len(lines)
host = codec._trim(cols, res).to_host()
for k in pj.COLS:
    assert np.array_equal(host[k], ref[k]), k
assert np.array_equal(el[: res.n_errors], el_r.cpu().numpy()) and np.array_equal(ec[: res.n_errors], ec_r.cpu().numpy())
codec.close()
print("pinned decode ok")
"""


@pytest.mark.parametrize("segment", [None, 1_000_003])
def test_host_decode_pinned_buffers(segment):
    """Input and output columns in pinned memory (pj_host_alloc) move by
    DMA with no bounce copy, one-shot and streamed: the columns, error lines
    and codes equal the device decode's."""
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.join(ROOT, "micronaut3-bug_amd"),
                                                      os.path.join(ROOT, "tests")]))
    if segment:
        env["PETJSON_DECODE_SEGMENT"] = str(segment)
    r = subprocess.run([sys.executable, "-c", PINNED], capture_output=True, text=True, env=env, timeout=240)
    assert r.returncode == 0 and "pinned decode ok" in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]


ARRAY_STREAM = r"""
import numpy as np, torch
import petjson as pj
codec = pj.Codec(0)
rng = np.random.default_rng(5)
els = []
for cfg, n in ((3, 30000), (5, 3000)):
    lines = codec.encode(pj.generate(cfg, n).to_device(), pj.FORMAT_NDJSON).cpu().numpy().tobytes().split(b"\n")[:-1]
    els += lines
# invalid elements that keep the frame: an unknown status, a missing name
for i in rng.choice(len(els), 300, replace=False):
    e = els[i]
    els[i] = e.replace(b'"status":"', b'"status":"x', 1) if i % 2 else e.replace(b'"name":', b'"nom":', 1)
# separators, brackets, quotes and backslashes inside strings; a 3 MB element
els.insert(7, b'{"name":"a,b],[c}{\\\\\\",","photoUrls":["[,]","\\\\"],"tags":[{"name":"]],,"}]}')
els.insert(20000, b'{"id":9,"name":"' + b"L" * 3_000_000 + b'","photoUrls":[],"status":"sold"}')
seps = [b",", b" ,\n  ", b",\n", b"\t,"]
doc = b" \n[" + b"".join(e + seps[j % 4] for j, e in enumerate(els[:-1])) + els[-1] + b"\n] \n"
d = torch.from_numpy(np.frombuffer(doc, np.uint8).copy()).cuda()
ref, el_r, ec_r, res_r = codec.decode(d, array=True)
ref = ref.to_host()
host, el, ec, res = codec.decode_array_host(doc)
assert res.n_lines == res_r.n_lines == len(els), (res.n_lines, res_r.n_lines, len(els))
for k in ("n_pets", "n_errors", "name_bytes", "cat_name_bytes", "n_urls", "url_bytes", "n_tags", "tag_name_bytes"):
    assert getattr(res, k) == getattr(res_r, k), (k, getattr(res, k), getattr(res_r, k))
for k in pj.COLS:
    assert np.array_equal(host[k], ref[k]), k
assert np.array_equal(el, el_r.cpu().numpy()) and np.array_equal(ec, ec_r.cpu().numpy())
# a broken frame is still a syntax error
try:
    codec.decode_array_host(doc.rsplit(b"]", 1)[0] + b"} \n")
    raise SystemExit("expected a syntax error")
except pj.PetJsonError as e:
    assert e.status == pj.PJ_ERR_SYNTAX, e
codec.close()
print("streamed array ok")
"""


@pytest.mark.parametrize("segment", [999_983, 4_194_301])
def test_host_array_document_streamed_in_segments(segment):
    """pj_decode_array_host on one JSON array document over
    PETJSON_DECODE_SEGMENT bytes decodes it in segments cut at top-level
    commas found on the device (separators, brackets and escapes inside
    strings, whitespace and newlines between elements, a 3 MB element longer
    than a segment, invalid elements): columns, element indices, codes and
    totals equal the one-shot device decode, and a broken frame is still
    PJ_ERR_SYNTAX."""
    env = dict(os.environ, PETJSON_DECODE_SEGMENT=str(segment),
               PYTHONPATH=os.pathsep.join([os.path.join(ROOT, "micronaut3-bug_amd"), os.path.join(ROOT, "tests")]))
    r = subprocess.run([sys.executable, "-c", ARRAY_STREAM], capture_output=True, text=True, env=env, timeout=240)
    assert r.returncode == 0 and "streamed array ok" in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]


ENC_STREAM = r"""
import ctypes as C
import numpy as np
import petjson as pj, oracle_py as orc
from model import from_columns, to_columns
codec = pj.Codec(0)
cases = [(1, 20000), (2, 40000), (3, 30000), (5, 4000)]
# a large record at a segment's first and last record
pets = from_columns(pj.generate(3, 3000), as_bytes=True)
for i in (0, 1499, 1500, 2999):
    pets[i].name = b"\x01\\\"" * 700
for cfg, n in cases + [(0, 0)]:
    cols = pj.generate(cfg, n) if cfg else to_columns(pets)
    for fmt in (pj.FORMAT_ARRAY, pj.FORMAT_NDJSON):
        want = orc.encode(cols, fmt)
        got = codec.encode_host(cols, fmt)
        assert got == want, (cfg, fmt, len(got), len(want))
        # capacity cut: the bytes before it may be written, none after it
        for cap in (len(want) - 1, len(want) // 2, 0):
            out = np.full(len(want) + 16, 0xEE, np.uint8)
            s, nn = cols.struct(), C.c_uint64(0)
            rc = codec.L.pj_encode_host(codec.ctx, C.byref(s), fmt, C.c_void_p(out.ctypes.data), cap, C.byref(nn))
            assert rc == pj.PJ_ERR_CAPACITY and nn.value == len(want), (cfg, fmt, cap, rc, nn.value)
            assert (out[cap:] == 0xEE).all(), (cfg, fmt, cap)
            w = out[:cap] != 0xEE
            ref = np.frombuffer(want, np.uint8)[:cap]
            assert (out[:cap][w] == ref[w]).all(), (cfg, fmt, cap)
    # pinned columns and output (pj_host_alloc): DMA with no bounce copy
    pc = pj.Columns(cols.n_pets, {}, dict(cols.caps))
    for k, v in cols.arrays.items():
        if v is None:
            pc.arrays[k] = None
            continue
        a = pj.host_array(len(v), v.dtype)
        a[:] = v
        pc.arrays[k] = a
    # the same pinned columns 8 bytes off 16-byte alignment
    pm = pj.Columns(cols.n_pets, {}, dict(cols.caps))
    for k, v in cols.arrays.items():
        if v is None:
            pm.arrays[k] = None
            continue
        raw = pj.host_array(v.nbytes + 16, np.uint8)
        a = raw[8: 8 + v.nbytes].view(v.dtype)
        a[:] = v
        pm.arrays[k] = a
    for fmt in (pj.FORMAT_ARRAY, pj.FORMAT_NDJSON):
        want = orc.encode(cols, fmt)
        out = pj.host_array(len(want) + 64, np.uint8)
        for cs in (pc, pm):
            s, nn = cs.struct(), C.c_uint64(0)
            rc = codec.L.pj_encode_host(codec.ctx, C.byref(s), fmt, C.c_void_p(out.ctypes.data), out.size, C.byref(nn))
            assert rc == pj.PJ_OK and out[: nn.value].tobytes() == want, (cfg, fmt, cs is pm, rc)
codec.close()
print("streamed encode ok")
"""


@pytest.mark.parametrize("segment,chunk", [(99_991, 0), (1_000_003, 65537), (0, 0)])
def test_host_encode_streamed_in_segments(segment, chunk):
    """pj_encode_host on columns over PETJSON_ENCODE_SEGMENT bytes encodes
    them in segments of records, each copied in while the one before it
    encodes and out while the one after it encodes: the bytes equal the
    oracle's in both framings (the array's brackets and separators across
    segment boundaries, large escape-heavy records at a segment's first and
    last record), a capacity cut writes nothing past it and reports the
    size needed, and pinned columns and output give the same bytes.
    segment 0: the default sizes, under which these inputs take the one-shot path."""
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.join(ROOT, "micronaut3-bug_amd"),
                                                      os.path.join(ROOT, "tests")]))
    if segment:
        env["PETJSON_ENCODE_SEGMENT"] = str(segment)
    if chunk:
        env["PETJSON_XFER_CHUNK"] = str(chunk)
    r = subprocess.run([sys.executable, "-c", ENC_STREAM], capture_output=True, text=True, env=env, timeout=240)
    assert r.returncode == 0 and "streamed encode ok" in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]


SMALL = r"""
import ctypes as C
import numpy as np
import petjson as pj, oracle_py as orc
codec = pj.Codec(0)
# column bytes from a few KiB to past 4 MiB (one launch to the bounce buffer
# below, the copy engine above), in ordinary and in pinned memory
for n in (0, 1, 3, 150, 400, 11000, 14000, 16000, 20000):
    text = np.frombuffer(orc.encode(pj.generate(3, n), pj.FORMAT_NDJSON) + b'{"name":1}\n{"name":"x","photoUrls":[]}', np.uint8)
    ref, rel, rec, rres = orc.decode(text.tobytes())
    for pinned in (False, True):
        mk = pj.host_array if pinned else (lambda k, dt: np.empty(k, dt))
        caps = {"cap_pets": rres.n_pets, "cap_name_bytes": rres.name_bytes, "cap_cat_name_bytes": rres.cat_name_bytes,
                "cap_urls": rres.n_urls, "cap_url_bytes": rres.url_bytes, "cap_tags": rres.n_tags,
                "cap_tag_name_bytes": rres.tag_name_bytes}
        size = {k: len(ref[k]) for k in pj.COLS}
        arr = {k: mk(size[k] + 1, pj.DTYPES[k]) for k in pj.COLS}
        for a in arr.values():
            a.view(np.uint8)[:] = 0xA5
        src = mk(text.size, np.uint8)
        src[:] = text
        el, ec = mk(4, np.uint64), mk(4, np.uint8)
        s, res = pj.Columns(0, arr, caps).struct(), pj.DecodeResult()
        rc = codec.L.pj_decode_host(codec.ctx, src.ctypes.data, src.size, C.byref(s), el.ctypes.data, ec.ctypes.data, 4,
                                    C.byref(res))
        assert rc == 0 and res.n_pets == rres.n_pets and res.n_errors == 1, (n, pinned, rc)
        assert el[0] == rel[0] and ec[0] == rec[0]
        for k in pj.COLS:
            assert np.array_equal(arr[k][:size[k]], ref[k]), (n, pinned, k)
            assert (arr[k][size[k]:].view(np.uint8) == 0xA5).all(), (n, pinned, k)
for n in (0, 1, 150, 5000, 40000):
    for model in (pj.MODEL_ORDER, pj.MODEL_USER):
        text = orc.encode_model(pj.generate_model(model, n, seed=n), pj.FORMAT_NDJSON)
        rc, ref, rel, rec, rres = orc.decode_model(model, text)
        got, el, ec, res = codec.decode_model_host(model, text)
        assert res.n_pets == rres.n_pets == n
        ref = ref.to_host()
        assert np.array_equal(got.present, ref.present)
        for a, b in zip(got.col + got.bytes, ref.col + ref.bytes):
            assert (a is None and b is None) or np.array_equal(a, b)
codec.close()
print("small copies ok")
"""


@pytest.mark.parametrize("chunk", [0, 4096, 100_000])
def test_host_decode_small_copies(chunk):
    """Host decodes whose bytes go through the bounce buffers in one launch,
    and those on the other side of that rule (by size, by the bounce buffers'
    own size), from and to ordinary and pinned memory, against the oracle; nothing is written past
    a column's end."""
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.join(ROOT, "micronaut3-bug_amd"), os.path.join(ROOT, "tests")]))
    if chunk:
        env["PETJSON_XFER_CHUNK"] = str(chunk)
    r = subprocess.run([sys.executable, "-c", SMALL], capture_output=True, text=True, env=env, timeout=240)
    assert r.returncode == 0 and "small copies ok" in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]
