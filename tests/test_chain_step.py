"""The rANS step that the chain kernels write out instruction by instruction, interpreted on
the CPU from the kernels' source: the table and the ring anywhere in LDS, against the step's
definition; and the wait states it has to hold itself, since the compiler looks into no asm."""
import os
import re

import numpy as np

from conftest import ROOT

SOURCE = os.path.join(ROOT, "gst_amd", "csrc", "gst_kernels.hip")
L = 1 << 15


def _step():
    """[(mnemonic, [operands])] of GST_CHAIN_STEP with its threshold and without its insertion."""
    text = open(SOURCE).read()
    body = re.search(r"#define GST_CHAIN_STEP\(THR, INSERT\)(.*?)\n  asm volatile", text, re.S).group(1)
    lines = "".join(re.findall(r'"(.*?)"', body.replace('" THR "', "%[thr]"))).split("\\n\\t")
    out = []
    for line in filter(None, lines):
        name, _, args = line.partition(" ")
        out.append((name, [a.strip().replace("%[", "").replace("]", "") for a in args.split(",")]
                    if name not in ("ds_read_b64", "s_waitcnt") else [args]))
    return out


def _interpret(step, lds, reg, lanes):
    """One step over the wave's registers `reg` (arrays for vector, integers for scalar ones)."""
    def val(a):
        return reg[a] if a in reg else int(a, 0)

    for name, args in step:
        if name == "ds_read_b64":
            addr = reg[re.fullmatch(r"v\[120:121\], %\[(\w+)\]", args[0]).group(1)]
            for k, dst in enumerate(("v120", "v121")):
                reg[dst] = np.array([int.from_bytes(lds[a + 4 * k:a + 4 * k + 4], "little") for a in addr])
            continue
        if name == "s_waitcnt":
            continue
        dst, a = args[0], [val(x) for x in args[1:]]
        if name == "v_cmp_lt_u32":
            mask = a[0] < a[1]
            reg["vcc"], reg["vcc_lo"] = mask, mask[:32]
            continue
        reg[dst] = {
            "v_and_b32": lambda: a[0] & a[1],
            "v_lshlrev_b32": lambda: a[1] << a[0],
            "v_lshrrev_b32": lambda: a[1] >> a[0],
            "v_lshl_add_u32": lambda: (a[0] << a[1]) + a[2],
            "v_mbcnt_lo_u32_b32": lambda: np.array([a[0][:i].sum() for i in range(lanes)]) + a[1],
            "v_cndmask_b32": lambda: np.where(a[2], a[1], a[0]),
            "s_bcnt1_i32_b32": lambda: int(a[0].sum()),
            "s_lshl3_add_u32": lambda: (a[0] << 3) + a[1],
            "v_mad_u32_u24": lambda: (a[0] & 0xFFFFFF) * (a[1] & 0xFFFFFF) + a[2],
        }[name]() & 0xFFFFFFFF


def test_step_takes_its_table_and_ring_from_any_lds_address():
    rng = np.random.default_rng(5)
    f = np.array([1793] + [1] * 255)
    sym = np.repeat(np.arange(256), f)
    off = np.arange(2048) - (np.cumsum(f) - f)[sym]
    words = rng.integers(0, 1 << 16, 256)
    s = words & 2047
    for table_at, ring_at in ((0, 16384), (256, 16640 + 6144), (40960, 8192)):
        lds = bytearray(rng.integers(0, 256, 65536, dtype=np.uint8).tobytes())
        table = np.stack([f[sym] | sym << 24, off], -1)
        ring = np.stack([f[sym[s]] << 5 | sym[s] << 24, (words >> 11) * f[sym[s]] + off[s]], -1)
        lds[table_at:table_at + 16384] = table.astype("<u4").tobytes()
        lds[ring_at:ring_at + 2048] = ring.astype("<u4").tobytes()
        y = rng.integers(0, 1 << 21, 32)
        y[::3] %= L
        assert 0 < (y < L).sum() < 32
        reg = {"y": y.copy(), "thr": np.full(32, L), "tab": table_at, "q": ring_at + 8 * 7}
        _interpret(_step(), lds, reg, 32)
        need = y < L
        at = 7 + np.cumsum(need) - need
        x = np.where(need, y << 16 | words[np.where(need, at, 0)], y)
        slot = x & 2047
        assert (reg["v120"] >> 24 == sym[slot]).all()
        assert (reg["y"] == (x >> 11) * f[sym[slot]] + off[slot]).all()
        assert reg["q"] == ring_at + 8 * (7 + need.sum())


def test_two_instructions_between_a_vector_write_of_a_mask_and_its_vector_read_as_a_number():
    names = [(n, " ".join(a)) for n, a in _step()]
    text = open(SOURCE).read()
    ans = re.search(r"#define GST_ANS_UPDATE(.*?)#define GST_ANS_OUT", text, re.S).group(1)
    for step in (names, [tuple(line.split(" ", 1)) for line in
                         "".join(re.findall(r'"(.*?)"', ans)).split("\\n\\t") if " " in line]):
        writes = [i for i, (n, a) in enumerate(step) if n.startswith("v_cmp") and "vcc" in a]
        reads = [i for i, (n, a) in enumerate(step) if n.startswith("v_") and re.search(r"vcc_(lo|hi)", a)]
        assert len(writes) == 1 and reads and reads[0] - writes[0] > 2
