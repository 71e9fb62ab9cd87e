"""Host-side check of qmm_lds_kernel's LDS layout (infer.net_amd/csrc/qmm.hip), CPU only.

The kernel's direct global->LDS copies (global_load_lds: lane L of a copy writes its 16 or 4
bytes at the wave-uniform LDS address + L * size) and its MFMA operand reads are restated
here from the kernel's index expressions, for every tile shape that is built (one matrix in
blocks of one to four 32-route tiles, and of four with two 32-row slabs a wave; gate and up in
eight waves with one, two and four tiles, of which three may be multiplied). The test
then checks what the kernel relies on:
* the copies of one step land inside their stage and never overlap (a block with fewer
  activation pieces than waves copies each by two waves, the same bytes to the same place);
* every operand byte a lane reads was written by that step's copies;
* and it is the byte the MFMA needs: weight row `wr`, codes 32h + 8j .. +7 of the K step
  for MFMA j in lane half h, and route slot n's activations 32h + 8j .. +7 likewise;
* the epilogue's accumulator layout covers each (row, route slot) of the tile exactly once;
* the SwiGLU exchange stays inside the stages and reaches the up wave of the same rows;
* the K ranges of a dense launch cover its steps once, their reads stay inside the row, and the
  sum pass reads each accumulator where its block stored it.
"""
import itertools

import pytest

# (bits, 32-route tiles copied, tiles multiplied, form, slabs a wave): the instances built. Forms:
# "one" matrix in four waves, "split": gate in waves 0-3 and up in waves 4-7.
SHAPES = ([(bits, nt, nt, "one", 1) for bits in (8, 5) for nt in (1, 2, 3, 4)] +
          [(bits, 4, 4, "one", 2) for bits in (8, 5)] +
          [(bits, nt, nt, "split", 1) for bits in (8, 5) for nt in (1, 2)] +
          [(5, 4, ntc, "split", 1) for ntc in (4, 3)])


def stage_layout(bits, nt, form, rs):
    split = form == "split"
    nw = 8 if split else 4
    tr = 128 * rs
    ab = 64 * bits // 8
    a_st = tr * ab
    nmat = 2 if split else 1
    bc = 32 * nt
    st = nmat * a_st + bc * 128
    aq = (2 if bits == 8 else 5) * rs
    nbw = 1 if 4 * nt < nw else 4 * nt // nw
    pw = min(4 * nt, nw)
    assert nbw * nw == 4 * nt or (nbw == 1 and nw % pw == 0)
    return dict(nw=nw, tr=tr, ab=ab, a_st=a_st, nmat=nmat, bc=bc, st=st, aq=aq, nbw=nbw, pw=pw, split=split)


def copies(bits, nt, form, rs):
    """LDS byte -> what it holds after one step's copies: ('w', matrix, row, byte) or
    ('x', route slot, element)."""
    L = stage_layout(bits, nt, form, rs)
    lds, times = {}, {}

    def put(addr, val, again=1):
        assert 0 <= addr < L["st"], (addr, L["st"])
        times[addr] = times.get(addr, 0) + 1
        assert times[addr] <= again and lds.get(addr, val) == val, ("two copies write one LDS byte", addr)
        lds[addr] = val

    for wave in range(L["nw"]):
        slab = wave & 3
        m = wave >> 2
        for q in range(L["aq"]):
            for lane in range(64):
                if bits == 8:
                    rl, sl = 16 * q + (lane >> 2), lane & 3
                    crow = slab * 32 * rs + rl
                    coff = 16 * (sl ^ ((rl >> 2) & 3))
                    dst = m * L["a_st"] + (slab * 32 * rs + 16 * q) * 64 + 16 * lane
                    for b in range(16):
                        put(dst + b, ("w", m, crow, coff + b))
                else:
                    i = 64 * q + lane
                    rl = i // 10
                    crow = slab * 32 * rs + rl
                    coff = 4 * (i - rl * 10)
                    dst = m * L["a_st"] + slab * 32 * rs * 40 + q * 256 + 4 * lane
                    for b in range(4):
                        put(dst + b, ("w", m, crow, coff + b))
        for i in range(L["nbw"]):
            piece = L["nw"] * i + wave % L["pw"]
            for lane in range(64):
                n = piece * 8 + (lane >> 3)
                sl = lane & 7
                src_el = 8 * (sl ^ ((n >> 1) & 7))
                dst = L["nmat"] * L["a_st"] + piece * 8 * 128 + 16 * lane
                for b in range(16):
                    put(dst + b, ("x", n, src_el + b // 2, b % 2), L["nw"] // L["pw"])
    return L, lds


@pytest.mark.parametrize("bits,nt,ntc,form,rs", SHAPES)
def test_operand_reads_see_their_copies(bits, nt, ntc, form, rs):
    L, lds = copies(bits, nt, form, rs)
    for wave in range(L["nw"]):
        slab = wave & 3
        m = wave >> 2
        for lane in range(64):
            r, h = lane & 31, lane >> 5
            # weights: the lane's chunk (codes 32h..32h+31 of row wr in this K step)
            for rsi in range(rs):
                wr = slab * 32 * rs + 32 * rsi + r
                if bits == 8:
                    sw = (r >> 2) & 3
                    ra = m * L["a_st"] + wr * 64
                    got = [lds[ra + 16 * ((2 * h) ^ sw) + b] for b in range(16)] + \
                          [lds[ra + 16 * ((2 * h + 1) ^ sw) + b] for b in range(16)]
                    want = [("w", m, wr, 32 * h + b) for b in range(32)]
                else:
                    ra = m * L["a_st"] + (wr * 10 + 5 * h) * 4
                    got = [lds[ra + b] for b in range(20)]
                    want = [("w", m, wr, 20 * h + b) for b in range(20)]
                assert got == want, (wave, lane, rsi, m)
            # activations: MFMA j reads route slot n's elements 32h + 8j .. +7
            bb = L["nmat"] * L["a_st"]
            for j in range(4):
                for i in range(ntc):
                    n = 32 * i + r
                    pc = 4 * h + j
                    addr = bb + n * 128 + 16 * (pc ^ ((n >> 1) & 7))
                    got = [lds[addr + b] for b in range(16)]
                    want = [("x", n, 32 * h + 8 * j + b // 2, b % 2) for b in range(16)]
                    assert got == want, (wave, lane, j, i)


@pytest.mark.parametrize("bits,nt,form,rs", sorted({(b, n, f, rs) for b, n, _, f, rs in SHAPES}))
def test_copies_fill_the_stage(bits, nt, form, rs):
    """Each step's copies write every byte of the weight rows and route slots."""
    L, lds = copies(bits, nt, form, rs)
    weights = sorted(v for v in lds.values() if v[0] == "w")
    want_w = sorted(("w", m, row, b) for m in range(L["nmat"]) for row in range(L["tr"]) for b in range(L["ab"]))
    assert weights == want_w
    acts = sorted(v for v in lds.values() if v[0] == "x")
    want_x = sorted(("x", n, e, half) for n in range(L["bc"]) for e in range(64) for half in range(2))
    assert acts == want_x
    assert 4 * L["st"] <= 160 * 1024


@pytest.mark.parametrize("nt,rs", [(1, 1), (2, 1), (3, 1), (4, 1), (4, 2)])
def test_epilogue_covers_each_output_once(nt, rs):
    """Accumulator element k of lane (r, h) in route tile i of a wave's slab is output row
    (wave * rs + slab) * 32 + 8*(k/4) + 4h + k%4 of the tile and route slot 32i + r (the
    32x32x16 MFMA's C layout), as the epilogue stores it."""
    seen = set()
    for wave, rsi, lane, i, q, k in itertools.product(range(4), range(rs), range(64), range(nt), range(4), range(4)):
        r, h = lane & 31, lane >> 5
        key = (wave * 32 * rs + 32 * rsi + 8 * q + 4 * h + k, 32 * i + r)
        assert key not in seen
        seen.add(key)
    assert len(seen) == 128 * rs * 32 * nt


@pytest.mark.parametrize("bits,nt,ntc", [(b, n, c) for b, n, c, form, _ in SHAPES if form == "split"])
def test_exchange_stays_inside_its_stage(bits, nt, ntc):
    """silu(gate) of slab s goes through stage s: element k of route tile i of a lane at float
    (16 i + k) * 64 + lane, where the up wave of the slab reads the same lane's."""
    L = stage_layout(bits, nt, "split", 1)
    for gate, up in zip(range(4), range(4, 8)):
        assert gate & 3 == up & 3
    at = [4 * ((16 * i + k) * 64 + lane) for i in range(ntc) for k in range(16) for lane in range(64)]
    assert len(set(at)) == len(at) and max(at) + 4 <= L["st"]


@pytest.mark.parametrize("columns,ranges", [(512, 1), (512, 2), (1536, 3), (2560, 4), (2560, 5), (4096, 8), (5120, 7),
                                            (7680, 4), (8192, 16), (8192, 32)])
def test_ranges_cover_the_steps_once(columns, ranges):
    """K ranges of a dense launch: whole four-step windows, the last range shorter where they do
    not divide; a window's scales (four groups of the row, one 8-byte load) and the copies
    issued ahead (clamped to the range's last step) stay inside the row."""
    G, S = columns // 64, 4
    ksteps = 4 * -(-(G // 4) // ranges)
    assert -(-G // ksteps) == ranges
    steps = []
    for rng in range(ranges):
        k0 = rng * ksteps
        nk = min(ksteps, G - k0)
        assert nk > 0 and nk % 4 == 0
        issued, kg = [], 0   # the kernel's issue(): S - 1 ahead, then one a step
        for _ in range(S - 1 + nk):
            issued.append(k0 + kg)
            kg += kg + 1 < nk
        for u in range(nk):
            assert issued[u] == k0 + u
        assert max(issued) < G
        for w in range(nk // 4):
            first = k0 + 4 * w
            assert first % 4 == 0 and first + 4 <= G and (2 * first) % 8 == 0
        steps += range(k0, k0 + nk)
    assert steps == list(range(G))


@pytest.mark.parametrize("rows,tokens,nt,ranges", [(128, 5, 1, 2), (300, 33, 1, 3), (129, 97, 2, 2), (513, 100, 3, 4)])
def test_sum_pass_reads_what_the_blocks_stored(rows, tokens, nt, ranges):
    """The accumulator quads of a plane: where a block of (range, row tile, chunk) stores lane
    (r, h)'s quad q of token tile i and slab w, and the (row, token) that splitk_sum_kernel
    takes from there, once each."""
    row_tiles, chunks = -(-rows // 128), -(-tokens // (32 * nt))
    quads = row_tiles * chunks * 1024 * nt   # of one plane
    assert quads % 256 == 0
    stored = {}
    for rng, rt, chunk in itertools.product(range(ranges), range(row_tiles), range(chunks)):
        at = ((rng * row_tiles + rt) * chunks + chunk) * (128 * 32 * nt)   # floats
        nvalid = min(32 * nt, tokens - chunk * 32 * nt)
        for w, i, q, lane in itertools.product(range(4), range(nt), range(4), range(64)):
            if 32 * i >= nvalid:
                continue
            quad = at // 4 + w * (nt * 4 * 64) + lane + (i * 4 + q) * 64
            assert quad not in stored and quad < ranges * quads
            stored[quad] = (rng, rt * 128 + w * 32 + 8 * q + 4 * (lane >> 5), (chunk * nt + i) * 32 + (lane & 31))
    seen = set()
    for f in range(quads):
        lane, g = f & 63, f >> 6
        q, g = g & 3, g >> 2
        i, g = g % nt, g // nt
        w, item = g & 3, g >> 2
        rt, chunk = item // chunks, item % chunks
        tok, row = (chunk * nt + i) * 32 + (lane & 31), rt * 128 + w * 32 + 8 * q + 4 * (lane >> 5)
        if tok >= tokens or row >= rows:
            continue
        assert [stored[rng * quads + f] for rng in range(ranges)] == [(rng, row, tok) for rng in range(ranges)]
        seen.add((row, tok))
    assert seen == {(row, tok) for row in range(0, rows, 4) for tok in range(tokens)}


def _tile_major_offsets(rows, rs, experts, G):
    """Byte offsets (into the tile-major copy) of every 4-byte piece the streaming kernel's
    copies read, padding rows included, and the (expert, row, piece offset, K step) each
    one belongs to. The copy pads an expert's rows to whole 256-row tiles (Matrix::tiled_rows);
    a copy lane's offset is tile * TR * row_bytes + (crow >> 7) * 128 * row_bytes +
    (crow & 127) * 40 + its piece offset, plus 128 * 40 per K step (qmm_lds_kernel)."""
    import numpy as np
    ab, row_bytes = 40, 40 * G
    rows_pad = (rows + 255) // 256 * 256
    tr = 128 * rs
    e, rt, slab, q, lane, kg = np.meshgrid(np.arange(experts), np.arange((rows + tr - 1) // tr), np.arange(4),
                                           np.arange(5 * rs), np.arange(64), np.arange(G), indexing="ij")
    i = 64 * q + lane
    rl = i // 10
    crow, coff = slab * 32 * rs + rl, 4 * (i - rl * 10)
    row = rt * tr + crow
    tpart = (crow >> 7) * 128 * row_bytes + (crow & 127) * ab + coff
    t_off = e * rows_pad * row_bytes + rt * tr * row_bytes + tpart + kg * 128 * ab
    return t_off, e, row, coff, kg, rows_pad


@pytest.mark.parametrize("rows,rs", [(256, 1), (200, 1), (384, 2), (300, 2), (129, 2)])
def test_tile_major_reads_match_row_major(rows, rs):
    """5-bit streaming launches read the codes from the tile-major copy that
    retile5_kernel writes ([expert][row tile][K step][row in tile][40 bytes], rows padded to
    whole 256-row tiles). Restates both index maps (the kernel's and the retile kernel's) on
    two experts and checks every byte a copy reads is the byte the row-major layout holds
    at row * row_bytes + K step * 40 + piece offset, for rows of the matrix, and zero
    padding inside the copy for the rows past it (their outputs are not stored)."""
    import numpy as np
    experts, G = 2, 8
    row_bytes = 40 * G
    t_off, e, row, coff, kg, rows_pad = _tile_major_offsets(rows, rs, experts, G)
    packed = np.arange(experts * rows * row_bytes, dtype=np.int64)   # byte b holds b
    words = packed.reshape(experts * rows, G, 10, 4)
    tiled = np.full(experts * rows_pad * row_bytes, -1, dtype=np.int64)
    for f in range(experts * rows):                                   # retile5_kernel
        ee, rr = divmod(f, rows)
        tile = ee * (rows_pad // 128) + rr // 128
        for k in range(G):
            for d in range(10):
                dst = ((tile * G + k) * 128 + rr % 128) * 10 + d
                tiled[4 * dst:4 * dst + 4] = words[f, k, d]
    assert t_off.min() >= 0 and t_off.max() + 4 <= tiled.size
    valid = row < rows
    r_off = (e * rows + row) * row_bytes + coff + kg * 40
    for b in range(4):
        assert np.array_equal(tiled[t_off[valid] + b], packed[r_off[valid] + b])
        assert (tiled[t_off[~valid] + b] == -1).all()


@pytest.mark.parametrize("rows", [16400, 16384 + 128, 16384 + 129, 4100, 300])
def test_tile_major_two_slab_copies_stay_in_bounds(rows):
    """Dense two-slab launches (256-row tiles) of single-expert 5-bit matrices: every byte
    a copy reads lies inside the tile-major copy, for rows % 256 in 1..128 (where 128-row
    padding would leave the last tile's upper slabs outside it) and above."""
    G = 8
    t_off, _, _, _, _, rows_pad = _tile_major_offsets(rows, 2, 1, G)
    tiled_bytes = rows_pad * 40 * G
    assert t_off.min() >= 0 and t_off.max() + 4 <= tiled_bytes
