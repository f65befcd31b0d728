"""What a program does with this framework, at the sizes it meets: one dict a case.

`path` names the public entry point a case goes through:

  load     LoadCompressedDXT / LoadRGB        one texture, staging buffer on the device
  loads    LoadCompressedDXTs / LoadRGBs      several textures in one staging buffer
  batch    Batch.decode, the plan bound before, or Batch.bind + Batch.decode each pass
  host     DecompressDXT                      .gtc bytes on the host in, DXT1 bytes out
  ans      AnsDecoder.decode                  stand-alone interleaved rANS groups, host to host
  serve    Server                             a burst of .gtc files from the host

Textures have legal sizes (both sides multiples of 128, whole rANS groups per plane).  Their
files come from the encoder at the benchmark's noise; a texture larger than one encoded
piece repeats the piece's rANS groups plane by plane, which keeps the symbol statistics,
the group sizes and a palette that grows with the texture, and takes a fraction of the time.
"""
import struct

import numpy as np
import torch

import gst_amd
from gst_amd import encode, serve

UNIT_TEXELS = 131072            # 16 x 8192: the smallest legal area
NOISE = 300                     # the encoder's default texture noise (thousandths)
MAX_TEXELS = 4096 * 4096
TABLE = 2048


def listed():
    return [
        # A single texture: the smallest legal one, a common one, one of no power of two
        # (an odd number of tiles a row), and the largest of the benchmark.
        {"name": "dxt_128x1024", "path": "load", "rgb": False, "sizes": "128x1024", "noise": NOISE},
        {"name": "dxt_512x512", "path": "load", "rgb": False, "sizes": "512x512", "noise": NOISE},
        {"name": "dxt_1920x1024", "path": "load", "rgb": False, "sizes": "1920x1024", "noise": NOISE},
        {"name": "dxt_4096x4096", "path": "load", "rgb": False, "sizes": "4096x4096", "noise": NOISE},
        # A page of equal thumbnails in one call, as the photo demo streams them.
        {"name": "dxts_page_16x512", "path": "loads", "rgb": False, "sizes": "512x512*16", "noise": NOISE},
        # RGB output for consumers that cannot sample DXT1: one preview, and a mixed page.
        {"name": "rgb_512x512", "path": "load", "rgb": True, "sizes": "512x512", "noise": NOISE},
        {"name": "rgbs_mixed_6", "path": "loads", "rgb": True,
         "sizes": "1024x1024*2,2048x1024,640x1024,512x512*2", "noise": NOISE},
        # Scene load: the benchmark's mix of 128 textures in one plan that stays bound.
        {"name": "batch_scene_128", "path": "batch", "rgb": False, "bind": False,
         "sizes": "512x512*32,1024x1024*32,512x1024*32,2048x2048*32", "noise": NOISE},
        # Streaming: another handful of uneven textures every frame, bound and decoded.
        {"name": "batch_bind_24", "path": "batch", "rgb": False, "bind": True,
         "sizes": "512x512*12,1024x1024*6,384x1024*2,1920x1024*2,2048x2048*2", "noise": NOISE},
        # A tool that turns a file in memory into DXT1 blocks in memory.
        {"name": "host_1024x1024", "path": "host", "rgb": False, "sizes": "1024x1024", "noise": NOISE},
        # The stand-alone rANS decoder on 24 groups of 32 interleaved streams.
        {"name": "ans_24x32", "path": "ans", "groups": 24, "streams": 32, "noise": NOISE},
        # The decode server: a burst of requests with their files on the host.
        {"name": "serve_burst_24", "path": "serve", "rgb": False,
         "sizes": "512x512*12,1024x1024*7,2048x2048*4,4096x4096", "noise": NOISE},
    ]


def _draw_size(rng, limit):
    """A legal size of about log-uniform area, of any legal aspect."""
    while True:
        area = UNIT_TEXELS * 2 ** rng.uniform(0, np.log2(limit / UNIT_TEXELS))
        w = 128 * max(1, round(2 ** rng.uniform(0, 5)))
        step = UNIT_TEXELS // np.gcd(UNIT_TEXELS, 128 * w)
        h = 128 * int(step) * max(1, round(area / (128 * int(step) * w)))
        if w * h <= limit and h <= 8192:
            return w, h


def draw(rng):
    path = rng.choice(["load", "load", "load", "loads", "loads", "batch", "batch", "host", "ans", "serve"])
    noise = rng.choice([100, 200, 300, 300, 300, 450])
    if path == "ans":
        return {"path": path, "groups": rng.randint(1, 128), "streams": rng.choice([32, 32, 24, 7, 1]),
                "noise": noise}
    rgb = path in ("load", "loads", "batch") and rng.random() < 0.35
    n = {"load": 1, "host": 1, "loads": round(2 ** rng.uniform(1, 5)), "batch": round(2 ** rng.uniform(1, 6)),
         "serve": rng.randint(4, 32)}[path]
    sizes = ["%dx%d" % _draw_size(rng, MAX_TEXELS if n <= 2 else 1 << 21) for _ in range(n)]
    case = {"path": path, "rgb": rgb, "sizes": ",".join(sizes), "noise": noise}
    if path == "batch":
        case["bind"] = rng.random() < 0.5
    return case


# ---- inputs ---------------------------------------------------------------------------

def _sizes(case):
    out = []
    for item in case["sizes"].split(","):
        size, _, times = item.partition("*")
        w, h = (int(v) for v in size.split("x"))
        out += [(w, h)] * int(times or 1)
    return out


def _split(gtc):
    """(header words, frequencies, [groups of bytes per stream]) of a .gtc file."""
    hdr = struct.unpack_from("<7I", gtc, 0)
    nv = hdr[0] * hdr[1] // 16
    at, streams = 28 + 2048, []
    for syms, size in zip((2 * nv, 4 * nv, hdr[2], nv), hdr[3:]):
        ends = np.frombuffer(gtc, "<u4", syms // 8192, at)
        starts = np.concatenate([[4 * len(ends)], ends[:-1]])
        streams.append([gtc[at + int(a):at + int(b)] for a, b in zip(starts, ends)])
        at += size
    return hdr, gtc[28:28 + 2048], streams


def _repeat(gtc, w, h):
    """The .gtc of a w x h texture whose planes repeat those of `gtc`."""
    hdr, freqs, streams = _split(gtc)
    times = w * h // (hdr[0] * hdr[1])
    if times == 1 and (w, h) == hdr[:2]:
        return gtc
    parts = []
    for groups, planes in zip(streams, (2, 4, 1, 1)):
        per = len(groups) // planes
        seq = [g for p in range(planes) for g in groups[p * per:(p + 1) * per] * times]
        ends = 4 * len(seq) + np.cumsum([len(g) for g in seq])
        parts.append(ends.astype("<u4").tobytes() + b"".join(seq))
    return struct.pack("<7I", w, h, hdr[2] * times, *(len(p) for p in parts)) + freqs + b"".join(parts)


def _files(case, seed):
    """The case's .gtc files: at most eight encoded pieces of each of two sizes behind them."""
    sizes = _sizes(case)
    kinds = [2 if w * h // UNIT_TEXELS % 2 == 0 else 1 for w, h in sizes]
    specs, slot = [], []
    count = {1: 0, 2: 0}
    for k in kinds:
        i = count[k] % 8
        count[k] += 1
        spec = (1000003 * (seed + 1) + 16 * i + k, 256 * k, 512)
        if spec not in specs:
            specs.append(spec)
        slot.append(specs.index(spec))
    pieces, _ = encode.make_textures(specs, noise_milli=case["noise"], want_dxt=False, encoder="gentenc")
    return [_repeat(pieces[s], w, h) for s, (w, h) in zip(slot, sizes)]


def _ans_inputs(case, seed):
    """Groups of interleaved streams with luma-like symbols: (frequencies, states, data)."""
    spec = [(1000003 * (seed + 1), 512, 512)]
    (gtc,), _ = encode.make_textures(spec, noise_milli=case["noise"], want_dxt=False, encoder="gentenc")
    freqs = np.frombuffer(gtc, "<u2", 256, 28).astype(np.int64)
    rng = np.random.default_rng(seed)
    groups, n = case["groups"], case["streams"]
    syms = rng.choice(256, size=(groups, n, 256), p=freqs / freqs.sum())
    cum = np.concatenate([[0], np.cumsum(freqs)[:-1]])
    x = np.full((groups, n), 1 << 15, np.int64)
    words = [[] for _ in range(groups)]
    for i in range(256):
        s = syms[:, :, i]
        f, c = freqs[s], cum[s]
        over = x >= f << 20
        for g in range(groups):
            if over[g].any():
                words[g].append((x[g][over[g]] & 0xFFFF).astype("<u2"))
        x = np.where(over, x >> 16, x)
        x = ((x // f) << 11) + x % f + c
    data = [np.concatenate(w).tobytes() if w else b"" for w in words]
    return freqs.tolist(), x.reshape(-1).tolist(), data


def _device(data):
    return torch.frombuffer(bytearray(data), dtype=torch.uint8).cuda()


def _out_bytes(hdr, rgb):
    return hdr.width * hdr.height * 3 if rgb else hdr.dxt_bytes


class _Memory:
    """Device memory the framework owns, as torch sees foreign memory."""

    def __init__(self, ptr, nbytes):
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (ptr, False), "version": 2}


def prepare(case, seed):
    gst_amd.InitializeDecoder(0)
    path = case["path"]
    state = {"path": path, "rgb": case.get("rgb", False)}
    if path == "ans":
        freqs, states, data = _ans_inputs(case, seed)
        state.update(decoder=gst_amd.AnsDecoder(freqs, case["streams"]), states=states, data=data)
        return state
    files = _files(case, seed)
    if path == "host":
        state["file"] = files[0]
    elif path in ("load", "loads"):
        staging, hdrs = gst_amd.PackStaging(files)
        total = sum(_out_bytes(h, state["rgb"]) for h in hdrs)
        state.update(hdrs=hdrs, cmp=_device(staging), out=torch.empty(total, dtype=torch.uint8, device="cuda"))
    elif path == "batch":
        hdrs = [gst_amd.ParseHeader(f) for f in files]
        total = sum(_out_bytes(h, state["rgb"]) for h in hdrs)
        out = torch.empty(total, dtype=torch.uint8, device="cuda")
        d_files = [_device(f) for f in files]
        ptrs, at = [], out.data_ptr()
        for h in hdrs:
            ptrs.append(at)
            at += _out_bytes(h, state["rgb"])
        batch = gst_amd.Batch(len(files), sum(h.num_blocks for h in hdrs), sum(h.palette_bytes for h in hdrs),
                              rgb=state["rgb"])
        state.update(hdrs=hdrs, files=d_files, ptrs=ptrs, out=out, batch=batch, bind=case["bind"])
        if not case["bind"]:
            batch.bind(hdrs, [f.data_ptr() for f in d_files], ptrs, torch.cuda.current_stream().cuda_stream)
    else:
        texels = sum(w * h for w, h in _sizes(case))
        state.update(files=files, server=serve.Server(
            hbm_budget_bytes=2 * texels, host_staging_bytes=1 << 26, slots=2, max_batch_images=len(files),
            max_batch_blocks=texels // 16, auto_release=False))
    return state


def run(state):
    path = state["path"]
    if path == "ans":
        return np.frombuffer(b"".join(state["decoder"].decode(state["states"], state["data"])), np.uint8)
    if path == "host":
        return np.frombuffer(gst_amd.DecompressDXT(state["file"]), np.uint8)
    if path == "serve":
        server = state["server"]
        for i, f in enumerate(state["files"]):
            server.submit(f, tag=i)
        server.drain()
        done = sorted(server.poll(), key=lambda c: c.tag)
        # The program keeps the textures in memory of its own and gives the server's back.
        outs = [torch.as_tensor(_Memory(c.d_output, c.output_bytes), device="cuda").clone() for c in done]
        torch.cuda.current_stream().synchronize()
        for c in done:
            server.release(c.ticket)
        return outs
    stream = torch.cuda.current_stream().cuda_stream
    if path == "batch":
        if state["bind"]:
            state["batch"].bind(state["hdrs"], [f.data_ptr() for f in state["files"]], state["ptrs"], stream)
        state["batch"].decode(stream)
    elif path == "load":
        load = gst_amd.LoadRGB if state["rgb"] else gst_amd.LoadCompressedDXT
        load(state["hdrs"][0], stream, state["cmp"].data_ptr(), state["out"].data_ptr())
    else:
        load = gst_amd.LoadRGBs if state["rgb"] else gst_amd.LoadCompressedDXTs
        load(state["hdrs"], stream, state["cmp"].data_ptr(), state["out"].data_ptr())
    return state["out"]


def work(case):
    """Compressed bytes read once (about 1.4 bits a texel at noise 100 to 450; the
    stand-alone groups about 2 bits a symbol) and output bytes written once.  The path is
    integer work: no floating-point operation is needed."""
    if case["path"] == "ans":
        return {"bytes": 256 * case["groups"] * case["streams"] * (1 + 2 / 8), "flops": 0}
    texels = sum(w * h for w, h in _sizes(case))
    return {"bytes": texels * (1.4 / 8 + (3 if case.get("rgb") else 0.5)), "flops": 0}


# ---- the results in plain numpy -----------------------------------------------------------

def _slots(freqs):
    freqs = np.asarray(freqs, np.int64)
    sym = np.repeat(np.arange(256), freqs)
    cum = np.concatenate([[0], np.cumsum(freqs)[:-1]])
    return sym, freqs[sym], np.arange(TABLE) - cum[sym]


def _rans(table, x, words, p):
    """256 steps of every group: states x[group, stream], its words below p[group]."""
    sym, f, off = table
    x, p = x.astype(np.int64), p.astype(np.int64)
    out = np.empty(x.shape + (256,), np.uint8)
    for i in range(255, -1, -1):
        slot = x & (TABLE - 1)
        out[:, :, i] = sym[slot]
        x = (x >> 11) * f[slot] + off[slot]
        need = x < 1 << 15
        total = need.sum(1)
        at = (p - total)[:, None] + np.cumsum(need, 1) - need
        x = np.where(need, (x << 16) | words[np.where(need, at, 0)], x)
        p = p - total
    return out


def _symbols(buf, groups, freqs):
    ends = np.frombuffer(buf, "<u4", groups).astype(np.int64)
    states = np.frombuffer(buf, "<u4", len(buf) // 4)
    x = states[(ends[:, None] // 4 - 32) + np.arange(32)]
    return _rans(_slots(freqs), x, np.frombuffer(buf, "<u2").astype(np.int64), ends // 2 - 64).reshape(-1)


def _lift(v, n):
    """One 1-D synthesis step along the last axis, of its first n entries."""
    half = n // 2

    def mirror(i):
        i = 2 * n - 2 - i if i >= n else i
        return abs(i)

    def div(s, d):
        return np.where(s < 0, -((-s) // d), s // d)

    lo, hi = v[..., :half], v[..., half:n]
    even = np.stack([lo[..., k] - div(hi[..., mirror(2 * k - 1) // 2] + hi[..., mirror(2 * k + 1) // 2] + 2, 4)
                     for k in range(half)], -1)
    odd = np.stack([hi[..., k] + div(even[..., k] + even[..., mirror(2 * k + 2) // 2], 2) for k in range(half)], -1)
    return np.stack([even, odd], -1).reshape(v.shape[:-1] + (n,))


def _plane(symbols, w, h):
    """One plane of blocks, tiles of 32 x 32 in raster order, through five levels."""
    t = symbols.reshape(-1, 32, 32).astype(np.int32) - 128
    for n in (2, 4, 8, 16, 32):
        sq = _lift(t[:, :n, :n], n)
        t[:, :n, :n] = _lift(sq.swapaxes(1, 2), n).swapaxes(1, 2)
    t = t.astype(np.int8).astype(np.int32)
    return t.reshape(h // 32, w // 32, 32, 32).swapaxes(1, 2).reshape(-1)


def _endpoint(y, co, cg):
    def half(s):
        return np.where(s < 0, -((-s) // 2), s // 2)
    t = y - half(cg)
    b = half(t - co)
    return b + co, cg + t, b


def _decode(gtc, rgb):
    hdr = struct.unpack_from("<7I", gtc, 0)
    w, h, pal_bytes = hdr[:3]
    bw, bh = w // 4, h // 4
    nv = bw * bh
    freqs = np.frombuffer(gtc, "<u2", 1024, 28).reshape(4, 256)
    at, syms = 28 + 2048, []
    for k, (count, size) in enumerate(zip((2 * nv, 4 * nv, pal_bytes, nv), hdr[3:])):
        syms.append(_symbols(gtc[at:at + size], count // 8192, freqs[k]))
        at += size
    y = [_plane(syms[0][i * nv:(i + 1) * nv], bw, bh) for i in range(2)]
    c = [_plane(syms[1][i * nv:(i + 1) * nv], bw, bh) for i in range(4)]
    word = syms[2].view("<u4")[np.cumsum(syms[3].astype(np.int64) - 128)].astype(np.int64)
    ends = [_endpoint(y[i], c[2 * i], c[2 * i + 1]) for i in range(2)]
    if not rgb:
        e = [((r << 11) | (g << 5) | b) & 0xFFFF for r, g, b in ends]
        out = np.empty((nv, 2), "<u4")
        out[:, 0] = e[0] | (e[1].astype(np.int64) << 16)
        out[:, 1] = word
        return out.reshape(-1).view(np.uint8)
    full = [np.stack([(r << 3) | (r >> 2), (g << 2) | (g >> 4), (b << 3) | (b >> 2)], -1) for r, g, b in ends]

    def third(s):
        return np.where(s < 0, -((-s) // 3), s // 3)
    pal = np.stack([full[0], full[1], third(2 * full[0] + full[1]), third(full[0] + 2 * full[1])], 1)
    sel = (word[:, None] >> (2 * np.arange(16))) & 3
    tex = pal[np.arange(nv)[:, None], sel].astype(np.uint8)  # block, texel, channel
    return tex.reshape(bh, bw, 4, 4, 3).swapaxes(1, 2).reshape(-1)


def exact(case, seed):
    if case["path"] == "ans":
        freqs, states, data = _ans_inputs(case, seed)
        n = case["streams"]
        ends = np.cumsum([len(d) // 2 for d in data])
        words = np.frombuffer(b"".join(data) + b"\0\0", "<u2").astype(np.int64)
        return _rans(_slots(freqs), np.array(states).reshape(-1, n), words, ends).reshape(-1)
    if sum(w * h for w, h in _sizes(case)) > 16 * MAX_TEXELS:
        return None  # too slow in numpy
    outs = [_decode(f, case.get("rgb", False)) for f in _files(case, seed)]
    return outs if case["path"] == "serve" else np.concatenate(outs)
