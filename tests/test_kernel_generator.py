"""CPU checks of the assembly that gen_eval_reg_kernel.py writes: the copies of tree blocks and border images
from global memory to LDS are followed through the straight-line part of every kernel (up to the tree loop) and
through one turn of the loop, and every source offset and LDS destination must stay inside what the host
allocates. A wrong step of the staging offset faults the GPU; here it fails an assertion."""
import importlib.util
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _generator():
    path = os.path.join(ROOT, "catboost_amd", "csrc", "gen_eval_reg_kernel.py")
    spec = importlib.util.spec_from_file_location("gen_eval_reg_kernel", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def _copies(lines, wave, lane, wave_bytes):
    """(source offset from the table's start, LDS address) of every global -> LDS copy of one lane, in order,
    and the index of the first copy of the tree loop."""
    s100 = wave * wave_bytes
    v2 = s28 = m0 = None
    copies, loop_at = [], None
    for line in lines:
        line = line.strip()
        if line.endswith("_loop:") and loop_at is None:
            loop_at = len(copies)
        if line.startswith("v_lshlrev_b32_e32 v2, 2, v1"):
            v2 = lane * 16
        found = re.match(r"s_sub_u32 s28, s100, (\d+)", line)
        if found:
            s28 = (s100 - int(found.group(1))) & 0xffffffff
        if line == "v_add_u32_e32 v2, s28, v2":
            v2 = (v2 + s28) & 0xffffffff
        found = re.match(r"v_add_u32_e32 v2, (0x[0-9a-f]+), v2", line)
        if found:
            v2 = (v2 + int(found.group(1), 16)) & 0xffffffff
        found = re.match(r"s_add_u32 m0, s100, (\d+)", line)
        if found:
            m0 = s100 + int(found.group(1))
        found = re.match(r"global_load_lds_dwordx4 v2, s\[26:27\](?: offset:(\d+))?", line)
        if found:
            offset = int(found.group(1) or 0)
            copies.append(((v2 + offset) & 0xffffffff, m0 + offset + lane * 16))
        if line.startswith("s_branch") and line.endswith("_loop"):
            break
    return copies, loop_at


@pytest.mark.parametrize("fused", [False, True])
def test_staging_copies_stay_inside_the_tables(fused):
    gen = _generator()
    if fused:
        cases = [(buckets, waves, 1, 256, False, six, True, levels) for buckets, waves in gen.FUSED_SHAPES
                 for six in (False, True)
                 for levels in ((None, 6) if buckets <= gen.FUSED_SIX_LEVEL_BUCKETS else (None,))]
    else:
        cases = [variant + (False, None) for variant in gen.VARIANTS]
    for buckets, waves, pitch, leaves, mixed, six, is_fused, levels in cases:
        text, _ = gen.gen_kernel(buckets, waves, pitch, leaves, mixed, six, fused=is_fused, levels=levels)
        lines = text.split("\n")
        block = gen.tree_block(pitch, leaves)
        buf_bytes = block * leaves * pitch * 8
        wave_bytes = buf_bytes // waves
        images = gen.fused_chunks(buckets, six) if is_fused else 0
        name = gen.kernel_name(buckets, waves, pitch, leaves, mixed, six, is_fused)
        for wave, lane in ((0, 0), (waves - 1, 63)):
            copies, loop_at = _copies(lines, wave, lane, wave_bytes)
            assert copies and loop_at is not None, name
            share = wave * wave_bytes + lane * 16
            # before the loop: the border images (fused kernels) and the first tree block, each in whole; in the loop
            # (one turn = two tree blocks) the two blocks behind the one being evaluated
            per_buffer = wave_bytes // 1024
            assert loop_at == (images + 1) * per_buffer, name
            for index, (source, lds) in enumerate(copies):
                assert 0 <= lds and lds + 16 <= 2 * buf_bytes, (name, index, lds)
                # a lane copies the same 16 bytes of its wave's share of a block into the same place of a buffer
                assert lds % buf_bytes == source % buf_bytes == share + (index % per_buffer) * 1024, (name, index, source, lds)
                # the table holds the images, the model's tree blocks and two blocks of null trees behind them;
                # up to the end of the loop's first turn the copies read the images and the first three blocks
                assert source < (images + 3) * buf_bytes, (name, index, source)
                assert source % 16 == 0 and (source % buf_bytes) // wave_bytes == wave, (name, index, source)
            # the blocks are read in order and each lands in the buffer that the kernel evaluates next
            staged = []
            for source, lds in copies:
                item = (source // buf_bytes, lds // buf_bytes)
                if not staged or staged[-1] != item:
                    staged.append(item)
            tail = staged[-3:]
            assert [b for b, _ in tail] == [images, images + 1, images + 2], (name, staged)
            assert [buffer for _, buffer in tail] == [0, 1, 0], (name, staged)
            if is_fused:
                assert [b for b, _ in staged[:images]] == list(range(images)), (name, staged)
                assert [buffer for _, buffer in staged[:images]] == [i % 2 for i in range(images)], (name, staged)


def _registers(text):
    """Scalar registers that an instruction's operands name."""
    found = set()
    for first, last in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        found.update(range(int(first), int(last) + 1))
    found.update(int(r) for r in re.findall(r"\bs(\d+)\b", text))
    return found


def _scalar_load_faults(lines, units):
    """Follows scalar loads, which return in any order, along every path of a kernel (of a fused kernel: every path of a
    model of `units` units, whose number sits in s28 while the rows are binarized): instructions that name a register
    which a load may still write, and loads into such a register."""
    code, label_at = [], {}
    for line in lines:
        line = line.strip()
        if line.startswith(".Lend"):
            break
        if line.endswith(":"):
            label_at[line[:-1]] = len(code)
        elif line and not line.startswith((".", ";", "#")):
            code.append(line)
    loop_at = next(at for label, at in label_at.items() if label.endswith("_loop"))
    # the loop's loads into s3 only pull lines into the cache: nothing reads the register there or behind it
    sink = re.compile(r"s_load_dword s3, ")
    assert not any(3 in _registers(c) for c in code[loop_at:] if not sink.match(c))
    unit_phase = [at for at, c in enumerate(code) if c == "s_mov_b32 s28, s89"]
    state = {0: frozenset()}  # registers with a load in flight on arrival at an instruction
    work, faults = [0], set()
    while work:
        at = work.pop()
        c, flying = code[at], state[at]
        op, _, operands = c.partition(" ")
        after, targets = flying, [at + 1]
        if op == "s_waitcnt":
            after = frozenset() if "lgkmcnt(0)" in c else flying
        elif op.startswith("s_load_"):
            destination = _registers(operands.split(",")[0])
            if _registers(operands) & flying:
                faults.add((at, c))
            after = flying if at >= loop_at and sink.match(c) else flying | destination
        elif op == "s_branch":
            targets = [label_at[operands]]
        elif op.startswith("s_cbranch"):
            targets.append(label_at[operands])
            compared = re.match(r"s_cmp_le_u32 s28, (\d+)$", code[at - 1])
            if units is not None and compared and unit_phase and at > unit_phase[0] and op == "s_cbranch_scc1":
                targets = [targets[1] if units <= int(compared.group(1)) else targets[0]]
        elif op == "s_endpgm":
            targets = []
        elif op.startswith(("s_", "v_", "ds_", "global_")):
            if _registers(operands) & flying:
                faults.add((at, c))
        else:
            raise AssertionError("unknown instruction: " + c)
        for target in targets:
            merged = after | state.get(target, frozenset())
            if target not in state or merged != state[target]:
                state[target] = merged
                work.append(target)
    return sorted(faults)


def test_scalar_loads_in_flight_keep_their_registers():
    """A record of a unit that the model lacks must have arrived before the record after next is requested into its
    registers: images with two such units in a row (one or two units beyond a multiple of four in the six-bit form)
    would otherwise binarize sixteen columns with whichever record came last."""
    gen = _generator()
    for variant in gen.VARIANTS:
        text, _ = gen.gen_kernel(*variant)
        assert not _scalar_load_faults(text.split("\n"), None), gen.kernel_name(*variant)
    for buckets, waves in gen.FUSED_SHAPES:
        for six in (False, True):
            for levels in (None, 6):
                text, _ = gen.gen_kernel(buckets, waves, 1, 256, False, six, fused=True, levels=levels)
                name = gen.kernel_name(buckets, waves, 1, 256, False, six, True, levels)
                for units in range(1, buckets // 16 + 1):
                    assert not _scalar_load_faults(text.split("\n"), units), (name, units)


@pytest.mark.parametrize("levels", [None, 6])
@pytest.mark.parametrize("six", [False, True])
def test_fused_kernels_of_columns(six, levels):
    """The column-major fused kernels: their copies follow the rows' ones, scalar loads keep their registers for any
    number of units, and every load goes to registers that no bin and no value in flight holds."""
    gen = _generator()
    for buckets, waves in gen.FUSED_COLUMN_SHAPES:
        text, _ = gen.gen_kernel(buckets, waves, 1, 256, False, six, fused=True, levels=levels, columns=True)
        lines = text.split("\n")
        name = gen.kernel_name(buckets, waves, 1, 256, False, six, True, levels, True)
        assert lines[1] == ".globl " + name
        wave_bytes = 32 * 1024 // waves
        images = gen.fused_chunks(buckets, six)
        rows_shape = next((b, w) for b, w in gen.FUSED_SHAPES if w == waves)
        rows, _ = gen.gen_kernel(*rows_shape, 1, 256, False, six, fused=True, levels=levels)
        for wave, lane in ((0, 0), (waves - 1, 63)):
            copies, loop_at = _copies(lines, wave, lane, wave_bytes)
            assert loop_at == (images + 1) * (wave_bytes // 1024), name
            share = wave * wave_bytes + lane * 16
            for index, (source, lds) in enumerate(copies):
                assert 0 <= lds and lds + 16 <= 64 * 1024 and source < (images + 3) * 32 * 1024, (name, index)
                assert lds % 32768 == source % 32768 == share + (index % (wave_bytes // 1024)) * 1024, (name, index)
            expected, _ = _copies(rows.split("\n"), wave, lane, wave_bytes)
            assert len(copies) - loop_at == len(expected) - (gen.fused_chunks(rows_shape[0], six) + 1) * (wave_bytes // 1024)
        for units in range(1, buckets // 16 + 1):
            assert not _scalar_load_faults(lines, units), (name, units)
        # every column of every unit is loaded once for each of the four documents, and waited for before its search reads it
        flying, loads, bins, aside = [], 0, set(), None
        for line in lines[:next(i for i, l in enumerate(lines) if l == name + "_loop:")]:
            line = line.strip()
            found = re.match(r"s_branch (%s_c\d+_end)$" % name, line)
            if found:  # what follows is jumped to from a turn's search, before the next loads
                aside = found.group(1) + ":"
            if aside is not None:
                aside = None if line == aside else aside
                continue
            found = re.match(r"global_load_dword v(\d+), v\d+, s\[30:31\] nt$", line)
            if found:
                register = int(found.group(1))
                assert register not in flying and register not in bins, (name, line)
                flying.append(register)
                loads += 1
            elif line.startswith("global_load_lds"):
                flying.append(None)
            elif "vmcnt(" in line:
                keep = int(re.search(r"vmcnt\((\d+)\)", line).group(1))
                del flying[:max(0, len(flying) - keep)]
            else:
                used = {int(r) for r in re.findall(r"\bv(\d+)\b", line)}
                for first, last in re.findall(r"\bv\[(\d+):(\d+)\]", line):
                    used.update(range(int(first), int(last) + 1))
                assert not used & set(flying), (name, line)
                found = re.match(r"v_lshrrev_b32_e32 v(\d+), 2, v(6|7|8|9)$", line)
                if found:
                    bins.add(int(found.group(1)))
        assert loads == buckets * 4 and len(bins) == buckets, (name, loads, len(bins))


def test_fused_kernels_of_columns_fetch_nothing_for_units_that_the_model_lacks():
    """The loads of every unit but the first run under a mask that is empty for a unit beyond the model's, and full again
    behind them."""
    gen = _generator()
    for buckets, waves in gen.FUSED_COLUMN_SHAPES:
        text, _ = gen.gen_kernel(buckets, waves, 1, 256, False, True, fused=True, columns=True)
        masked, unit_loads = None, {}
        for line in (line.strip() for line in text.split("\n")):
            found = re.match(r"s_cmp_gt_u32 s28, (\d+)$", line)
            if found:
                masked = int(found.group(1))
            elif line == "s_mov_b64 exec, -1":
                masked = None
            elif line.startswith("global_load_dword v") and line.endswith(" nt"):
                unit_loads[masked] = unit_loads.get(masked, 0) + 1
        # (the first unit, which every model has, is loaded without a mask)
        assert unit_loads == {unit or None: 64 for unit in range(buckets // 16)}
        assert text.count("s_cselect_b64 exec, -1, 0") == text.count("s_mov_b64 exec, -1")


def test_only_the_fused_kernels_of_rows_start_late():
    gen = _generator()
    for columns, shapes in ((False, gen.FUSED_SHAPES), (True, gen.FUSED_COLUMN_SHAPES)):
        for buckets, waves in shapes:
            text, _ = gen.gen_kernel(buckets, waves, 1, 256, False, True, fused=True, columns=columns)
            assert ("s_sleep" in text) == (not columns)


def _signed(byte):
    return byte - 256 if byte >= 128 else byte


def _places(code, scalars, bins, bins_at, weight):
    """Follows one lane through the vector instructions of a tree (up to its first leaf gather) and gives the LDS offsets that
    the gathers of the four documents name. `bins`: dwords of the bins registers from register `bins_at` on. Also checks what
    the hardware asks for: two instructions between the last write of the product's index and the product, five between the
    product and the first gather, no vector register in src0 of anything but a level's compare in index mode."""
    v = {bins_at + i: dword for i, dword in enumerate(bins)}
    index, written, product_at, gathers = None, {}, None, []
    bytes_of = lambda x: [(x >> (8 * j)) & 255 for j in range(4)]  # noqa: E731
    dword = lambda b: sum(x << (8 * j) for j, x in enumerate(b))   # noqa: E731

    def value(operand):
        if operand.startswith("v"):
            return v[int(operand[1:])]
        return scalars[int(operand[1:])] if operand.startswith("s") else int(operand, 0)

    masks = [m.group(1) for m in (re.match(r"v_bitop3_b32 v\d+, v(\d+),", c) for c in code) if m]
    lows = [m.group(1) for m in (re.match(r"v_bitop3_b32 v3, v(\d+),", c) for c in code) if m]
    low = int(lows[0])
    v[int(next(m for m in masks if int(m) != low))], v[low] = 0x80808080, 0xc0c0c0c0
    for fold in (re.match(r"v_bitop3_b32 v3, v4, v(\d+), v3 bitop3:0x6a$", c) for c in code):
        if fold:
            v[int(fold.group(1))] = 0x7c7c7c7c if len(scalars) == 12 else 0x7f7f7f7f
    for at, c in enumerate(code):
        op, _, rest = c.partition(" ")
        args = [x.strip() for x in rest.split(",")]
        if op == "s_set_gpr_idx_on":
            index = scalars[int(args[0][1:])] & 255
        elif op == "s_set_gpr_idx_idx":
            index = scalars[int(args[0][1:])] & 255
        elif op == "s_set_gpr_idx_off":
            index = None
        elif op in ("v_add_u32_e64", "v_lerp_u8"):
            assert index is not None and int(args[1][1:]) == bins_at
            a, b = bytes_of(v[bins_at + index]), bytes_of(value(args[2]))
            sums = [x + y for x, y in zip(a, b)]
            assert op == "v_lerp_u8" or max(sums) < 256
            v[int(args[0][1:])] = dword([x >> 1 for x in sums]) if op == "v_lerp_u8" else dword(sums)
            written[int(args[0][1:])] = at
        elif op.startswith(("v_bitop3", "v_lshrrev", "v_and_b32")):
            assert index is None
            if op.startswith("v_bitop3"):
                last, table = args[3].split()
                table = int(table.split(":")[1], 16)
                x, y, z = value(args[1]), value(args[2]), value(last)
                out = sum(((table >> (((x >> b & 1) << 2) | ((y >> b & 1) << 1) | (z >> b & 1))) & 1) << b for b in range(32))
            elif op.startswith("v_lshrrev"):
                out = value(args[2]) >> int(args[1])
            else:
                out = value(args[1]) & value(args[2])
            v[int(args[0][1:])] = out
            written[int(args[0][1:])] = at
        elif op.startswith("v_mfma"):
            assert at - written[3] > 2 and index is None
            first = int(re.match(r"v\[(\d+):", args[0]).group(1))
            for j in range(4):
                v[first + j] = weight * _signed(bytes_of(v[3])[j])
            product_at = at
        elif op.startswith("ds_read"):
            assert at - product_at > 5
            found = re.match(r"ds_read_b(64|128) v\[\d+:\d+\], v(\d+) offset:(\d+)$", c)
            gathers.append(v[int(found.group(2))] + int(found.group(3)))
        else:
            assert op in ("s_waitcnt", "s_nop", "v_add_f64", "s_load_dwordx16"), c
    return gathers


@pytest.mark.parametrize("shape", [(128, 4, 1, 64), (96, 8, 1, 64), (200, 4, 1, 256), (104, 4, 3, 64), (56, 4, 6, 64), (160, 4, 4, 256)])
@pytest.mark.parametrize("six", [False, True])
def test_places_of_leaf_values(shape, six):
    """The levels' compares, their merges and the product, followed for one lane: the gathers name the leaves that comparing
    bins with splits gives, at the edges of what the compare holds (bins and splits of 1 and 127 or 63, a bin of 128 or 64,
    a level that stands for none: constant 0, true for that bin alone)."""
    import random
    gen = _generator()
    buckets, waves, pitch, leaves = shape
    text, _ = gen.gen_kernel(buckets, waves, pitch, leaves, False, six)
    lines = [line.strip() for line in text.split("\n")]
    start = next(i for i, line in enumerate(lines) if line.endswith("_loop:")) + 1
    dims = 2 if leaves > 64 and pitch > 1 else 1  # of a piece of the table
    gathers = 4 * pitch // dims
    code = []
    for line in lines[start:]:
        code.append(line)
        if sum(c.startswith("ds_read") for c in code) == gathers:
            break
    depth, top = (6 if leaves == 64 else 8), (64 if six else 128)
    bins_at = int(re.search(r"v_add_u32_e64 v\d+, v(\d+), s", text).group(1))
    weight = 8 * dims >> (8 - depth)
    rng = random.Random(7)
    for _ in range(200):
        bins = [[rng.choice([0, 1, top // 2, top - 1, top, rng.randrange(top + 1)]) for _ in range(4)] for _ in range(buckets)]
        scalars, expected = {}, [0] * 4
        for d in range(depth):
            bucket, split = rng.randrange(buckets), rng.choice([1, 2, top - 1, top, rng.randrange(1, top + 1)])
            scalars[32 + 2 * d] = bucket
            scalars[33 + 2 * d] = ((64 if six and d % 2 == 0 else 128) - split) * 0x01010101
            for j in range(4):
                expected[j] |= int(bins[bucket][j] >= split) << d
        got = _places(code, scalars, [sum(x << (8 * j) for j, x in enumerate(b)) for b in bins], bins_at, weight)
        # (several dimensions: a leaf's place is the levels' results, each but the last one compared with the next; the top one comes inverted)
        places = [x ^ (x >> 1) ^ (leaves >> 2) if pitch > 1 else x for x in expected]
        assert got == [8 * dims * x + k * leaves * 8 for x in places for k in range(0, pitch, dims)]


@pytest.mark.parametrize("shape", [(104, 4, 3, 64), (56, 4, 6, 64), (192, 4, 2, 64)])
def test_places_of_leaf_values_in_tables_that_are_not_folded(shape):
    """The other walk of the kernels of several dimensions and 64 leaves (trees of five levels and less), and the one kernel that has no other."""
    import random
    gen = _generator()
    buckets, waves, pitch, leaves = shape
    text, _ = gen.gen_kernel(buckets, waves, pitch, leaves, False, False)
    lines = [line.strip() for line in text.split("\n")]
    both = any(line.endswith("_plain:") for line in lines)
    assert both == (buckets != 192) and sum(line.endswith("_plain") for line in lines) == (3 if both else 0)  # two ways in, and its own turns
    code = []
    for line in lines[next(i for i, line in enumerate(lines) if line.endswith("_plain:" if both else "_loop:")) + 1:]:
        code.append(line)
        if sum(c.startswith("ds_read") for c in code) == 4 * pitch:
            break
    bins_at = int(re.search(r"v_add_u32_e64 v\d+, v(\d+), s", text).group(1))
    rng = random.Random(3)
    for _ in range(50):
        bins = [[rng.randrange(129) for _ in range(4)] for _ in range(buckets)]
        scalars, expected = {}, [0] * 4
        for d in range(6):
            bucket, split = rng.randrange(buckets), rng.randrange(1, 129)
            scalars[32 + 2 * d], scalars[33 + 2 * d] = bucket, (128 - split) * 0x01010101
            for j in range(4):
                expected[j] |= int(bins[bucket][j] >= split) << d
        got = _places(code, scalars, [sum(x << (8 * j) for j, x in enumerate(b)) for b in bins], bins_at, 2)
        assert got == [8 * x + k * 512 for x in expected for k in range(pitch)]


@pytest.mark.parametrize("shape", [(160, 4, 4, 64), (56, 4, 6, 64), (128, 4, 6, 64)])
@pytest.mark.parametrize("six", [False, True])
def test_places_of_leaf_values_in_pieces_of_two_dimensions(shape, six):
    """The third walk of the kernels of four and six dimensions and 64 leaves (trees of four levels and less): 16 bytes per leaf, not folded;
    the product's weight and the way in follow the same flag. Kernels of two and three dimensions have none."""
    import random
    gen = _generator()
    buckets, waves, pitch, leaves = shape
    text, _ = gen.gen_kernel(buckets, waves, pitch, leaves, False, six)
    assert all("_pairs" not in gen.gen_kernel(b, 4, p, n, False, six)[0] for b, p, n in ((104, 3, 64), (80, 2, 64), (192, 2, 64), (160, 4, 256)))
    lines = [line.strip() for line in text.split("\n")]
    assert sum(line.endswith("_pairs") for line in lines) == 3  # two ways in, and its own turns
    assert all(lines[i - 1] == "s_bitcmp1_b32 s15, 5" for i, line in enumerate(lines) if re.match(r"s_cbranch_scc1 .*_pairs$", line))
    at = lines.index("s_cselect_b32 s24, 4, 2")
    assert lines[at - 1] == "s_bitcmp1_b32 s15, 5" and re.match(r"v_lshlrev_b32_e64 v\d+, v5, s24$", lines[at + 1])
    code = []
    for line in lines[next(i for i, line in enumerate(lines) if line.endswith("_pairs:")) + 1:]:
        code.append(line)
        if sum(c.startswith("ds_read") for c in code) == 2 * pitch:
            break
    assert all(c.startswith("ds_read_b128") for c in code if c.startswith("ds_read"))
    bins_at = int(re.search(r"v_add_u32_e64 v\d+, v(\d+), s", text).group(1))
    top = 64 if six else 128
    rng = random.Random(5)
    for _ in range(50):
        bins = [[rng.randrange(top + 1) for _ in range(4)] for _ in range(buckets)]
        scalars, expected = {}, [0] * 4
        for d in range(6):
            bucket, split = rng.randrange(buckets), rng.randrange(1, top + 1)
            scalars[32 + 2 * d], scalars[33 + 2 * d] = bucket, ((64 if six and d % 2 == 0 else 128) - split) * 0x01010101
            for j in range(4):
                expected[j] |= int(bins[bucket][j] >= split) << d
        got = _places(code, scalars, [sum(x << (8 * j) for j, x in enumerate(b)) for b in bins], bins_at, 4)
        assert got == [16 * x + k * 512 for x in expected for k in range(0, pitch, 2)]


def _follow(lines, start, scalars, v, bins_at, weight):
    """As _places, for the trees that branch or have more than eight levels: follows a lane from line `start` on, branches taken as the
    scalars say, up to the next tree's first instruction behind the gathers, and gives the LDS offsets that they name. `v`: the vector
    registers' dwords. In index mode src0 may be a vector register in nothing but a level's read of its bucket."""
    labels = {line[:-1]: i for i, line in enumerate(lines) if line.endswith(":")}
    index, scc, step, product_step, gathers = None, 0, 0, None, []
    written = {}
    at = start

    def value(operand):
        if operand.startswith("v"):
            return v[int(operand[1:])]
        return scalars[int(operand[1:])] if operand.startswith("s") else int(operand, 0)

    while True:
        line = lines[at]
        at += 1
        if line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        args = [x.strip() for x in rest.split(",")]
        if gathers and not op.startswith("ds_read"):
            return gathers
        step += 1
        if op.startswith("s_set_gpr_idx_o") or op == "s_set_gpr_idx_idx":
            index = None if op.endswith("off") else scalars[int(args[0][1:])] & 255
        elif op == "s_bitcmp1_b32":
            scc = scalars[int(args[0][1:])] >> int(args[1]) & 1
        elif op in ("s_branch", "s_cbranch_scc1"):
            at = labels[args[0]] if op == "s_branch" or scc else at
        elif op.startswith("v_mfma"):
            assert step - written[3] > 2 and index is None
            first = int(re.match(r"v\[(\d+):", args[0]).group(1))
            for j in range(4):
                v[first + j] = weight * _signed(v[3] >> (8 * j) & 255)
            product_step = step
        elif op == "v_mul_u32_u24_sdwa":
            word = int(args[2].split()[-1][-1])
            v[int(args[0][1:])] = scalars[int(args[1][1:])] * (v[int(args[2].split()[0][1:])] >> (16 * word) & 0xffff)
        elif op.startswith("ds_read"):
            assert product_step is None or step - product_step > 5
            found = re.match(r"ds_read_b(64|128) v\[\d+:\d+\], v(\d+) offset:(\d+)$", line)
            gathers.append(v[int(found.group(2))] + int(found.group(3)))
        elif op in ("s_waitcnt", "s_nop", "v_add_f64", "s_load_dwordx16"):
            continue
        else:
            last, _, table = args[-1].partition(" ")
            sources = args[1:-1] + [last]
            if index is not None and sources[0].startswith("v"):
                assert op in ("v_add_u32_e64", "v_lerp_u8", "v_xor_b32_e64") and sources[0] == "v%d" % bins_at
                sources[0] = "v%d" % (bins_at + index)
            x = [value(s) for s in sources]
            if op in ("v_add_u32_e64", "v_lerp_u8"):
                sums = [(x[0] >> (8 * j) & 255) + (x[1] >> (8 * j) & 255) for j in range(4)]
                out = sum((s >> 1 if op == "v_lerp_u8" else s) << (8 * j) for j, s in enumerate(sums))
                assert op == "v_lerp_u8" or max(sums) < 256
            elif op == "v_subrev_u32_e32":
                out = (x[1] - x[0]) & 0xffffffff
            elif op == "v_bitop3_b32":
                truth = int(table.split(":")[1], 16)
                out = sum((truth >> ((x[0] >> b & 1) << 2 | (x[1] >> b & 1) << 1 | x[2] >> b & 1) & 1) << b for b in range(32))
            elif op == "v_bfi_b32":
                out = (x[0] & x[1]) | (~x[0] & x[2] & 0xffffffff)
            elif op == "v_perm_b32":
                both = x[1] | x[0] << 32  # selectors 0 to 3: bytes of the second operand, 4 to 7: of the first
                out = sum((both >> (8 * (x[2] >> (8 * j) & 7)) & 255) << (8 * j) for j in range(4))
            else:
                out = {"v_xor_b32_e64": lambda: x[0] ^ x[1], "v_or_b32_e32": lambda: x[0] | x[1], "v_and_b32_e32": lambda: x[0] & x[1],
                       "v_lshrrev_b32_e32": lambda: x[1] >> x[0]}[op]()
            v[int(args[0][1:])] = out
            written[int(args[0][1:])] = step


def _constants(lines, end):
    """Scalar and vector registers that hold a constant where the walk starts (the last move to each)."""
    scalars, v = {}, {}
    for line in lines[:end]:
        found = re.match(r"(s_mov_b32 s|v_mov_b32_e32 v)(\d+), (0x[0-9a-f]+|\d+)$", line)
        if found:
            (scalars if found.group(1)[0] == "s" else v)[int(found.group(2))] = int(found.group(3), 0)
    return scalars, v


@pytest.mark.parametrize("shape", [(96, 8, 1, 64), (208, 4, 1, 256), (56, 4, 6, 64), (104, 4, 3, 64), (192, 4, 2, 64), (160, 4, 4, 256)])
def test_places_of_leaf_values_of_mixed_trees(shape):
    """Both forms of a mixed kernel's tree: bit 31 of its first dword clear (pairs of levels) and set (eight bits a level, with and without a
    xor mask, splits on both sides of 128, and levels that stand for none: splitIdx 255), in every walk that the kernel has."""
    import random
    gen = _generator()
    buckets, waves, pitch, leaves = shape
    lines = [line.strip() for line in gen.gen_kernel(buckets, waves, pitch, leaves, True)[0].split("\n")]
    depth = 6 if leaves == 64 else 8
    rng = random.Random(11)
    walks = [i for i, line in enumerate(lines) if re.search(r"_(loop|plain|pairs):$", line)]
    assert len(walks) == (3 if leaves == 64 and pitch in (4, 6) else 2 if leaves == 64 and pitch == 3 else 1)
    for start in walks:
        folded = lines[start].endswith("_loop:") and pitch > 1 and buckets != 192
        dims = 2 if pitch > 1 and (leaves == 256 or lines[start].endswith("_pairs:")) else 1
        constants, vectors = _constants(lines, start)
        bins_at = next(int(m.group(1)) for m in (re.match(r"v_xor_b32_e64 v3, v(\d+), s", line) for line in lines) if m)
        for turn in range(120):
            wide = turn % 2 == 1
            top = 255 if wide else 128
            bins = [[rng.choice([0, 1, 127, 128, top, rng.randrange(top + 1)]) % (top + 1) for _ in range(4)] for _ in range(buckets)]
            scalars, expected = dict(constants), [0] * 4
            for d in range(depth):
                bucket = rng.randrange(buckets)
                split = rng.choice([1, 2, 127, 128, 129, 254, 255, rng.randrange(1, 256)]) if wide else rng.choice([1, 127, 128, rng.randrange(1, 129)])
                mask = rng.choice([0, 0, rng.randrange(256)]) if wide else 0
                if wide:
                    scalars.update({32 + 4 * d: bucket | (0x80000000 if d == 0 else 0), 33 + 4 * d: mask * 0x01010101,
                                    34 + 4 * d: (256 - split) * 0x01010101})
                else:
                    scalars.update({32 + 2 * d: bucket, 33 + 2 * d: (128 - split) * 0x01010101})
                for j in range(4):
                    expected[j] |= int(bins[bucket][j] ^ mask >= split) << d
            v = dict(vectors)
            v.update({bins_at + i: sum(x << (8 * j) for j, x in enumerate(b)) for i, b in enumerate(bins)})
            got = _follow(lines, start, scalars, v, bins_at, 8 * dims >> (8 - depth))
            places = [x ^ (x >> 1) ^ (leaves >> 2) if folded else x for x in expected]
            assert got == [8 * dims * x + k * leaves * 8 for x in places for k in range(0, pitch, dims)]


@pytest.mark.parametrize("shape", [(96, 8, 1, 1024), (208, 4, 1, 1024)])
@pytest.mark.parametrize("six", [False, True])
def test_places_of_leaf_values_of_ten_levels(shape, six):
    """Trees of depth 9 and 10: the ninth and tenth level join the eight merged in pairs, whose top bit is not inverted there."""
    import random
    gen = _generator()
    buckets, waves, pitch, leaves = shape
    lines = [line.strip() for line in gen.gen_kernel(buckets, waves, pitch, leaves, False, six)[0].split("\n")]
    start = next(i for i, line in enumerate(lines) if line.endswith("_loop:"))
    bins_at = next(int(m.group(1)) for m in (re.match(r"v_add_u32_e64 v\d+, v(\d+), s", line) for line in lines[start:]) if m)
    constants, vectors = _constants(lines, start)
    top = 64 if six else 128
    rng = random.Random(13)
    for _ in range(120):
        bins = [[rng.choice([0, 1, top - 1, top, rng.randrange(top + 1)]) for _ in range(4)] for _ in range(buckets)]
        scalars, expected = dict(constants), [0] * 4
        for d in range(10):
            bucket, split = rng.randrange(buckets), rng.choice([1, 2, top - 1, top, rng.randrange(1, top + 1)])
            scalars.update({32 + 2 * d: bucket, 33 + 2 * d: ((64 if six and d % 2 == 0 and d < 8 else 128) - split) * 0x01010101})
            for j in range(4):
                expected[j] |= int(bins[bucket][j] >= split) << d
        v = dict(vectors)
        v.update({bins_at + i: sum(x << (8 * j) for j, x in enumerate(b)) for i, b in enumerate(bins)})
        assert _follow(lines, start, scalars, v, bins_at, 8) == [8 * x for x in expected]


def test_the_hosts_table_says_how_the_kernels_read_their_leaves():
    """Leaf tables are laid out on the host by the table that the generator writes: which kernels fold them, and which have the walk of
    pieces of two dimensions, has to be what the kernels' instructions do; those of exchange kernels likewise."""
    gen = _generator()
    rows = re.findall(r'\{(\d+), (\d+), (\d+), (\d+), (\w+), (\w+), (\w+), (\w+), "(\w+)"\}', gen.generate_tables())
    assert len(rows) == len(gen.VARIANTS) and [int(r[0]) for r in rows] == sorted(int(r[0]) for r in rows)
    for buckets, waves, pitch, leaves, mixed, six, folds, pairs, name in rows:
        text, _ = gen.gen_kernel(int(buckets), int(waves), int(pitch), int(leaves), mixed == "true", six == "true")
        assert name + "_loop:" in text
        assert ("bitop3:0x6a" in text) == (folds == "true") and (name + "_pairs:" in text) == (pairs == "true")
        assert (name + "_plain:" in text) == (folds == "true" and leaves == "64")
        assert pitch != "1" or folds == pairs == "false"
    found = re.search(r"ExchangeFoldsLeaves\(int depth\) \{ return (.*); \}", gen.generate_tables()).group(1)
    exchange = gen.gen_eval_exchange_kernel
    for depth, six, fused in {(shape + (False,))[:3] for shape in exchange.SHAPES}:
        folded = exchange.folds_leaves(depth)
        assert folded == ("depth == %d" % depth in found.split(" || "))
        assert ("bitop3:0x6a" in exchange.gen_kernel(depth, six, fused, folded=folded)[0]) == folded
    with open(os.path.join(ROOT, "catboost_amd", "csrc", "hip_evaluator.hip")) as f:
        host = f.read()
    assert '#include "eval_reg_tables.inc"' in host and "cbamd_eval_reg_b" not in host and host.count("ExchangeFoldsLeaves(") == 1
