"""CPU checks of the exchange kernels: the assembly that gen_eval_exchange_kernel.py writes is run, instruction by
instruction, on the tables that exchange_plan.cpp makes for small random models. Every access must stay inside its table or LDS
area, no register or LDS byte may be used while a load into it is still under way, the waves of a workgroup run one behind the
other from barrier to barrier in changing orders, and the sums must be those of the documented order, bit for bit."""
import importlib.util
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "catboost_amd", "csrc")


def _generator():
    spec = importlib.util.spec_from_file_location("gen_eval_exchange_kernel", os.path.join(CSRC, "gen_eval_exchange_kernel.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("plan") / "exchange_plan_main")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", os.path.join(ROOT, "tests", "exchange_plan_main.cpp"),
                           os.path.join(CSRC, "exchange_plan.cpp"), "-o", out])
    return out


def _plan(planner, path, trees, buckets, max_depth, six, tiles=None):
    """tiles: (column of every bucket, byte offsets of the pieces, the columns) for a fused kernel."""
    with open(path, "w") as f:
        f.write("%d %d %d %d %d\n" % (len(trees), buckets, max_depth, six, len(tiles[1]) // 16 if tiles else 0))
        if tiles:
            f.write(" ".join(map(str, tiles[0])) + "\n")
        for levels, leaves in trees:
            f.write("%d\n" % len(levels))
            for bucket, split, one_hot in levels:
                add, xor = (1, ~split & 0x7f) if one_hot else (128 - split, 0)
                f.write("%d %d %d %d %g\n" % (bucket, add, xor, one_hot, abs(split / 60.0 - 0.5)))
            f.write(" ".join("%.17g" % v for v in leaves) + "\n")
        if tiles:
            f.write(" ".join(map(str, tiles[1])) + "\n")
            for used, one_hot, row_byte, values in tiles[2]:
                f.write("%d %d %d %d %s\n" % (used, one_hot, row_byte, len(values), " ".join(map(str, values))))
    lines = subprocess.check_output([planner, path], text=True).split("\n")
    if lines[0] == "refused":
        return None
    tables = [np.array(line.split(), dtype=np.uint32) for line in lines[1:4]]
    plan = (int(lines[0]), tables[0], tables[1], tables[2], np.array(lines[4].split(), dtype=np.float64))
    return plan + tuple(np.array(line.split(), dtype=np.uint32) for line in lines[5:7]) if tiles else plan


def _model(rng, tree_count, buckets, depths, bins_limit, one_hot_share, skew=False):
    trees = []
    for _ in range(tree_count):
        levels = []
        for _ in range(int(rng.choice(depths))):
            bucket = int(rng.integers(0, buckets))
            if skew and rng.random() < 0.6:
                bucket = int(rng.integers(0, 3))
            levels.append((bucket, int(rng.integers(1, bins_limit + 1)), bool(rng.random() < one_hot_share)))
        trees.append((levels, rng.normal(size=1 << len(levels))))
    return trees


def _expected(trees, bins):
    """Sixteen partial sums, a wave's pairs of trees in order, the odd last tree with wave 0; then the sums in order."""
    parts = np.zeros((16, bins.shape[0]))
    for t, (levels, leaves) in enumerate(trees):
        index = np.zeros(bins.shape[0], dtype=np.int64)
        for d, (bucket, split, one_hot) in enumerate(levels):
            b = bins[:, bucket].astype(np.int64)
            index |= (b == split if one_hot else b >= split).astype(np.int64) << d
        wave = 0 if len(trees) % 2 and t == len(trees) - 1 else t // 2 % 16
        parts[wave] += leaves[index]
    total = parts[0].copy()
    for wave in range(1, 16):
        total += parts[wave]
    return total


class _Memory:
    """Named byte arrays at made-up addresses; every access has to lie in one of them."""

    def __init__(self):
        self.areas = []

    def add(self, data):
        base = (len(self.areas) + 1) << 32
        self.areas.append((base, data))
        return base

    def at(self, address, size):
        base, data = self.areas[(address >> 32) - 1]
        offset = address - base
        assert 0 <= offset and offset + size <= len(data), (hex(address), size, len(data))
        return data, offset


class _Wave:
    def __init__(self, kernel, memory, lds, kernarg, group, wave):
        self.code, self.labels = kernel
        self.memory, self.lds = memory, lds
        self.s = [0] * 128
        self.v = np.zeros((128, 64), dtype=np.uint32)
        self.s[0], self.s[1], self.s[2] = kernarg & 0xffffffff, kernarg >> 32, group
        self.v[0] = np.arange(64) + 64 * wave
        self.pc, self.scc, self.vcc, self.m0, self.indexed = 0, 0, 0, 0, False
        self.exec = (1 << 64) - 1
        self.lgkm, self.vm = [], []          # (destination registers, finish) in flight
        self.flying = set()

    # -- operands
    def pair(self, text):
        first = int(re.match(r"s\[(\d+):", text).group(1))
        return self.s[first] | self.s[first + 1] << 32

    def scalar(self, text):
        if text == "m0":
            return self.m0
        if re.match(r"s\d+$", text):
            return self.s[int(text[1:])]
        return int(text, 0) & 0xffffffff

    def set_scalar(self, text, value):
        value &= 0xffffffff
        if text == "m0":
            self.m0 = value
        elif text == "exec_hi":
            self.exec = (self.exec & 0xffffffff) | value << 32
        else:
            self.s[int(text[1:])] = value

    def vector(self, text, first=False):
        if re.match(r"v\d+$", text):
            r = int(text[1:])
            if first and self.indexed and self.m0 >> 12 & 1:
                r += self.m0 & 0xff
                assert 64 <= r < 128
            return self.v[r]
        return np.uint32(self.scalar(text))

    def double(self, text):
        kind, first = re.match(r"([sv])\[(\d+):", text).groups()
        first = int(first)
        if kind == "s":
            return np.array([self.s[first], self.s[first + 1]], dtype=np.uint32).view(np.float64)[0]
        return np.stack([self.v[first], self.v[first + 1]], axis=1).copy().view(np.float64)[:, 0]

    @staticmethod
    def registers(text):
        out = set()
        for kind, first, last in re.findall(r"\b([sv])\[(\d+):(\d+)\]", text):
            out.update((kind, r) for r in range(int(first), int(last) + 1))
        out.update((kind, int(r)) for kind, r in re.findall(r"\b([sv])(\d+)\b", text))
        return out

    def issue(self, queue, destination, finish):
        self.flying |= destination
        queue.append((destination, finish))

    def land(self, queue, keep):
        while len(queue) > keep:
            destination, finish = queue.pop(0)
            finish()
            self.flying -= destination

    # -- runs to the next barrier; True at the end of the program
    def run(self):
        while True:
            op, args, text = self.code[self.pc]
            self.pc += 1
            if op == "s_endpgm":
                assert not self.lgkm and not [d for d, _ in self.vm if d]
                return True
            if op == "s_barrier":
                assert not [d for d, _ in self.lgkm if not d or min(d)[0] == "v"], "a barrier with LDS requests under way"
                return False
            if op != "s_waitcnt":
                assert not (self.registers(text) & self.flying), text
            getattr(self, "op_" + re.sub(r"_e32$|_e64$", "", op))(args)

    def op_s_waitcnt(self, args):
        text = " ".join(args)
        found = re.search(r"vmcnt\((\d+)\)", text)
        if found:
            self.land(self.vm, int(found.group(1)))
        if "lgkmcnt(0)" in text:
            self.land(self.lgkm, 0)

    def op_s_nop(self, args):
        pass

    def _s_load(self, args, count):
        first = int(re.match(r"s\[?(\d+)", args[0]).group(1))
        assert first % min(count, 4) == 0
        data, at = self.memory.at(self.pair(args[1]) + int(args[2], 0), 4 * count)
        values = [int(x) for x in data[at:at + 4 * count].view(np.uint32)]

        def finish():
            self.s[first:first + count] = values
        self.issue(self.lgkm, {("s", r) for r in range(first, first + count)}, finish)

    def op_s_load_dwordx2(self, args):
        self._s_load(args, 2)

    def op_s_load_dwordx4(self, args):
        self._s_load(args, 4)

    def op_s_load_dwordx8(self, args):
        self._s_load(args, 8)

    def op_s_load_dwordx16(self, args):
        self._s_load(args, 16)

    def op_s_mov_b32(self, args):
        self.set_scalar(args[0], self.scalar(args[1]))

    def op_s_cselect_b32(self, args):
        self.set_scalar(args[0], self.scalar(args[1] if self.scc else args[2]))

    def op_s_mov_b64(self, args):
        if args[0] == "exec":
            self.exec = (1 << 64) - 1 if args[1] == "-1" else self.pair(args[1])
            return
        to, source = (int(re.match(r"s\[(\d+):", a).group(1)) for a in args)
        self.s[to:to + 2] = self.s[source:source + 2]

    def op_s_add_u32(self, args):
        total = self.scalar(args[1]) + self.scalar(args[2])
        self.scc = total >> 32
        self.set_scalar(args[0], total)

    def op_s_addc_u32(self, args):
        total = self.scalar(args[1]) + self.scalar(args[2]) + self.scc
        self.scc = total >> 32
        self.set_scalar(args[0], total)

    def op_s_sub_u32(self, args):
        self.set_scalar(args[0], self.scalar(args[1]) - self.scalar(args[2]))

    def op_s_mul_i32(self, args):
        self.set_scalar(args[0], self.scalar(args[1]) * self.scalar(args[2]))

    def op_s_mul_hi_u32(self, args):
        self.set_scalar(args[0], self.scalar(args[1]) * self.scalar(args[2]) >> 32)

    def op_s_lshl_b32(self, args):
        self.set_scalar(args[0], self.scalar(args[1]) << self.scalar(args[2]))

    def op_s_lshr_b32(self, args):
        self.set_scalar(args[0], self.scalar(args[1]) >> self.scalar(args[2]))

    def op_s_and_b32(self, args):
        self.set_scalar(args[0], self.scalar(args[1]) & self.scalar(args[2]))

    def op_s_bfe_u32(self, args):
        spec = int(args[2], 0)
        self.set_scalar(args[0], self.scalar(args[1]) >> (spec & 31) & ((1 << (spec >> 16)) - 1))

    def op_s_cmp_eq_u32(self, args):
        self.scc = int(self.scalar(args[0]) == self.scalar(args[1]))

    def op_s_cmp_lg_u32(self, args):
        self.scc = int(self.scalar(args[0]) != self.scalar(args[1]))

    def op_s_cmp_gt_u32(self, args):
        self.scc = int(self.scalar(args[0]) > self.scalar(args[1]))

    def op_s_bitcmp1_b32(self, args):
        self.scc = self.scalar(args[0]) >> self.scalar(args[1]) & 1

    def op_s_branch(self, args):
        self.pc = self.labels[args[0]]

    def op_s_cbranch_scc1(self, args):
        if self.scc:
            self.pc = self.labels[args[0]]

    def op_s_load_dword(self, args):
        self._s_load(args, 1)

    def op_s_min_u32(self, args):
        self.set_scalar(args[0], min(self.scalar(args[1]), self.scalar(args[2])))

    def op_s_cmp_lt_u32(self, args):
        self.scc = int(self.scalar(args[0]) < self.scalar(args[1]))

    def op_s_cmp_ge_u32(self, args):
        self.scc = int(self.scalar(args[0]) >= self.scalar(args[1]))

    def op_v_subrev_u32(self, args):
        self._set(args, self.vector(args[2]) - self.vector(args[1], True))

    def op_v_min_u32(self, args):
        self._set(args, np.minimum(self.vector(args[1], True), self.vector(args[2])))

    def op_v_or_b32(self, args):
        self._set(args, self.vector(args[1], True) | self.vector(args[2]))

    def op_v_sub_u32(self, args):
        self._set(args, self.vector(args[1], True) - self.vector(args[2]))

    def op_v_mul_u32_u24(self, args):
        self._set(args, self.vector(args[1], True) * self.vector(args[2]))

    op_v_mul_lo_u32 = op_v_mul_u32_u24

    def op_v_lshl_add_u32(self, args):
        self._set(args, (self.vector(args[1], True) << self.vector(args[2])) + self.vector(args[3]))

    def op_v_lshl_or_b32(self, args):
        self._set(args, (self.vector(args[1], True) << self.vector(args[2])) | self.vector(args[3]))

    def op_v_lshrrev_b32_sdwa(self, args):
        # the low byte of the result into one byte of the destination, the others stay
        words = args[2].split()
        byte = int(re.match(r"dst_sel:BYTE_(\d)", words[1]).group(1))
        assert words[2:] == ["dst_unused:UNUSED_PRESERVE", "src0_sel:DWORD", "src1_sel:DWORD"]
        value = (self.vector(words[0]) >> self.vector(args[1])) & np.uint32(255)
        register = int(args[0][1:])
        self.v[register] = self.v[register] & np.uint32(~(255 << 8 * byte) & 0xffffffff) | value << np.uint32(8 * byte)

    def _floats(self, text):
        return np.asarray(self.vector(text), dtype=np.uint32).view(np.float32)

    def op_v_fma_f32(self, args):
        last, _, clamp = args[3].partition(" ")
        with np.errstate(all="ignore"):
            a, b, c = (self._floats(x).astype(np.float64) for x in (args[1], args[2], last))
            value = (a * b + c).astype(np.float32)
            if clamp:
                value = np.where(value > 0, np.minimum(value, np.float32(1)), np.float32(0)).astype(np.float32)
        self._set(args, value.view(np.uint32))

    def op_v_cmp_lt_f32(self, args):
        assert args[0] == "vcc"
        with np.errstate(all="ignore"):
            self.vcc = sum(1 << int(i) for i in np.flatnonzero(self._floats(args[1]) < self._floats(args[2])))

    def op_v_cmp_eq_u32(self, args):
        self.vcc = sum(1 << int(i) for i in np.flatnonzero(self.vector(args[1]) == self.vector(args[2])))

    def op_v_cndmask_b32(self, args):
        assert args[3] == "vcc"
        taken = np.array([self.vcc >> lane & 1 for lane in range(64)], dtype=bool)
        self._set(args, np.where(taken, self.vector(args[2]), self.vector(args[1])))

    def op_s_cbranch_scc0(self, args):
        if not self.scc:
            self.pc = self.labels[args[0]]

    def op_s_set_gpr_idx_on(self, args):
        self.indexed = True
        self.m0 = self.m0 & ~0xf0ff | self.scalar(args[0]) & 0xff | int(args[1], 0) << 12

    def op_s_set_gpr_idx_idx(self, args):
        assert self.indexed
        self.m0 = self.m0 & ~0xff | self.scalar(args[0]) & 0xff

    def op_s_set_gpr_idx_off(self, args):
        self.indexed = False

    def op_s_and_saveexec_b64(self, args):
        self.exec &= self.vcc

    def op_v_readfirstlane_b32(self, args):
        self.set_scalar(args[0], int(self.vector(args[1])[0]))

    def _set(self, args, value):
        assert self.exec == (1 << 64) - 1
        self.v[int(args[0][1:])] = value

    def op_v_mov_b32(self, args):
        if self.indexed and self.m0 >> 12 & 8:       # the destination is relative
            register = int(args[0][1:]) + (self.m0 & 0xff)
            assert 64 <= register < 128
            self.v[register] = self.vector(args[1])
        else:
            self._set(args, self.vector(args[1], True))

    def op_v_and_b32(self, args):
        self._set(args, self.vector(args[1], True) & self.vector(args[2]))

    def op_v_xor_b32(self, args):
        self._set(args, self.vector(args[1], True) ^ self.vector(args[2]))

    def op_v_add_u32(self, args):
        self._set(args, self.vector(args[1], True) + self.vector(args[2]))

    def op_v_lshrrev_b32(self, args):
        self._set(args, self.vector(args[2]) >> self.vector(args[1], True))

    def op_v_lshlrev_b32(self, args):
        self._set(args, self.vector(args[2]) << self.vector(args[1], True))

    def op_v_bfi_b32(self, args):
        mask = self.vector(args[1], True)
        self._set(args, (mask & self.vector(args[2])) | (~mask & self.vector(args[3])))

    def op_v_dot4_u32_u8(self, args):
        a, b = self.vector(args[1], True), self.vector(args[2])
        total = np.zeros(64, dtype=np.uint32) + self.vector(args[3])
        for j in range(4):
            total = total + ((a >> np.uint32(8 * j)) & np.uint32(255)) * ((b >> np.uint32(8 * j)) & np.uint32(255))
        self._set(args, total)

    def _set_double(self, args, value):
        first = int(re.match(r"v\[(\d+):", args[0]).group(1))
        words = np.ascontiguousarray(value).view(np.uint32).reshape(64, 2)
        self.v[first], self.v[first + 1] = words[:, 0], words[:, 1]

    def op_v_add_f64(self, args):
        self._set_double(args, self.double(args[1]) + self.double(args[2]))

    def op_v_mul_f64(self, args):
        self._set_double(args, self.double(args[1]) * self.double(args[2]))

    def op_v_cmp_ge_u32(self, args):
        first = int(re.match(r"s\[(\d+):", args[0]).group(1))
        mask = sum(1 << int(i) for i in np.flatnonzero(self.vector(args[1]) >= self.vector(args[2])))
        self.s[first:first + 2] = [mask & 0xffffffff, mask >> 32]

    def op_v_bfe_u32(self, args):
        self._set(args, self.vector(args[1], True) >> self.vector(args[2]) & np.uint32((1 << int(args[3])) - 1))

    def op_v_cmp_gt_u32(self, args):
        hit = self.vector(args[1]) > self.vector(args[2])
        self.vcc = sum(1 << int(i) for i in np.flatnonzero(hit))

    # -- LDS: reads look at the bytes when they are issued (requests of a wave stay in order)
    def _lds(self, address, size):
        assert (address % size == 0).all() and (address + size <= len(self.lds.data)).all(), address
        assert not self.lds.flying[address].any(), "LDS bytes that a copy still writes"
        return (address[:, None] + np.arange(size)[None, :]).astype(np.int64)

    @staticmethod
    def _offset(args):
        found = re.search(r"offset:(\d+)", " ".join(args))
        assert not found or int(found.group(1)) < 65536
        return int(found.group(1)) if found else 0

    def _ds_read(self, args, words):
        first = int(re.match(r"v\[?(\d+)", args[0]).group(1))
        address = self.vector(args[1].split()[0]).astype(np.int64) + self._offset(args)
        data = self.lds.data[self._lds(address, 4 * words)].copy().view(np.uint32).reshape(64, words)

        def finish():
            for i in range(words):
                self.v[first + i] = data[:, i]
        self.issue(self.lgkm, {("v", r) for r in range(first, first + words)}, finish)

    def op_ds_read_b32(self, args):
        self._ds_read(args, 1)

    def op_ds_read_b64(self, args):
        self._ds_read(args, 2)

    def op_ds_read_b128(self, args):
        self._ds_read(args, 4)

    def op_ds_read_u8(self, args):
        register = int(args[0][1:])
        address = self.vector(args[1].split()[0]).astype(np.int64) + self._offset(args)
        data = self.lds.data[self._lds(address, 1)][:, 0].astype(np.uint32)

        def finish():
            self.v[register] = data
        self.issue(self.lgkm, {("v", register)}, finish)

    def _ds_write(self, args, words):
        first = int(re.match(r"v\[?(\d+)", args[1]).group(1))
        lanes = [lane for lane in range(64) if self.exec >> lane & 1]
        address = self.vector(args[0]).astype(np.int64)[lanes] + self._offset(args)
        where = self._lds(address, 4 * words)
        data = np.stack([self.v[first + i][lanes] for i in range(words)], axis=1).copy().view(np.uint8).reshape(len(lanes), 4 * words)
        self.lds.data[where] = data                  # a wave's later requests find it there, other waves' behind a barrier
        self.issue(self.lgkm, set(), lambda: None)

    def op_ds_write_b32(self, args):
        self._ds_write(args, 1)

    def op_ds_write_b64(self, args):
        self._ds_write(args, 2)

    # the lane's dword at M0
    def op_ds_read_addtid_b32(self, args):
        register = int(args[0].split()[0][1:])
        address = (self.m0 & 0xffff) + self._offset(args) + 4 * np.arange(64)
        data = self.lds.data[self._lds(address, 4)].copy().view(np.uint32)[:, 0]

        def finish():
            self.v[register] = data
        self.issue(self.lgkm, {("v", register)}, finish)

    def op_ds_write_addtid_b32(self, args):
        address = (self.m0 & 0xffff) + self._offset(args) + 4 * np.arange(64)
        self.lds.data[self._lds(address, 4)] = self.v[int(args[0].split()[0][1:])].copy().view(np.uint8).reshape(64, 4)
        self.issue(self.lgkm, set(), lambda: None)

    # -- global memory
    def op_global_load_dwordx4(self, args):
        first = int(re.match(r"v\[(\d+):", args[0]).group(1))
        base = self.pair(args[2].split()[0]) + self._offset(args)
        values = self.v[first:first + 4].copy()
        for lane in range(64):
            if self.exec >> lane & 1:
                data, at = self.memory.at(base + int(self.vector(args[1])[lane]), 16)
                values[:, lane] = data[at:at + 16].copy().view(np.uint32)

        def finish():
            self.v[first:first + 4] = values
        self.issue(self.vm, {("v", r) for r in range(first, first + 4)}, finish)

    def op_global_load_dword(self, args):
        register = int(args[0][1:])
        base = self.pair(args[2].split()[0]) + self._offset(args)
        values = []
        for lane in range(64):
            data, at = self.memory.at(base + int(self.vector(args[1])[lane]), 4)
            values.append(data[at:at + 4].view(np.uint32)[0])

        def finish():
            self.v[register] = np.array(values, dtype=np.uint32)
        self.issue(self.vm, {("v", register)}, finish)

    def op_global_load_lds_dwordx4(self, args):
        base, offset = self.pair(args[1].split()[0]), self._offset(args)
        assert offset < 4096
        chunks = []
        for lane in range(64):
            if self.exec >> lane & 1:
                data, at = self.memory.at(base + int(self.vector(args[0])[lane]) + offset, 16)
                to = self.m0 + offset + 16 * lane
                assert 0 <= to and to + 16 <= len(self.lds.data)
                chunks.append((to, data[at:at + 16].copy()))
                self.lds.flying[to:to + 16] = True

        def finish():
            for to, data in chunks:
                self.lds.data[to:to + 16] = data
                self.lds.flying[to:to + 16] = False
        self.issue(self.vm, set(), finish)

    def op_global_store_dwordx2(self, args):
        first = int(re.match(r"v\[(\d+):", args[1]).group(1))
        base = self.pair(args[2])
        for lane in range(64):
            if self.exec >> lane & 1:
                data, at = self.memory.at(base + int(self.vector(args[0])[lane]), 8)
                data[at:at + 8] = self.v[first:first + 2, lane].copy().view(np.uint8)


class _Lds:
    def __init__(self, size, rng):
        self.data = rng.integers(0, 256, size=size).astype(np.uint8)  # LDS holds anything at first
        self.flying = np.zeros(size, dtype=bool)


def _kernel(gen, depth, six, fused=False):
    text, _ = gen.gen_kernel(depth, six, fused)
    code, labels = [], {}
    for line in text.split("\n"):
        line = line.strip()
        if line.startswith(".Lend"):
            break
        if line.endswith(":"):
            assert line[:-1] not in labels
            labels[line[:-1]] = len(code)
        elif line and not line.startswith("."):
            op, _, rest = line.partition(" ")
            code.append((op, [a.strip() for a in rest.split(",")] if rest else [], line))
    return code, labels


def _run(gen, plan, bins, doc_count, buckets, depth, six, scale, bias, rng, rows=None):
    """rows: the documents for a fused kernel, whose bins nobody gives it."""
    rounds, wave_table, records, extra_rows, leaves = plan[:5]
    blocks = bins.shape[0] // 256
    # [block][bucket][lane][j] with document = block * 256 + j * 64 + lane
    tiled = np.ascontiguousarray(bins.reshape(blocks, 4, 64, buckets).transpose(0, 3, 2, 1)).reshape(-1).view(np.uint8)
    memory = _Memory()
    out = np.full(doc_count, np.nan)
    addresses = [memory.add(np.ascontiguousarray(a).view(np.uint8)) for a in
                 (tiled, wave_table, records, extra_rows, leaves, out, np.array([bias]))]
    kernarg = np.zeros(112, dtype=np.uint8)
    kernarg[:56] = np.array(addresses, dtype=np.uint64).view(np.uint8)
    kernarg[56:64] = np.array([scale]).view(np.uint8)
    kernarg[64:80] = np.array([doc_count, rounds, buckets * 256, 0], dtype=np.uint32).view(np.uint8)
    if rows is not None:
        fused = [memory.add(np.ascontiguousarray(a).reshape(-1).view(np.uint8)) for a in (rows, plan[5], plan[6])]
        kernarg[80:96] = np.array(fused[:2], dtype=np.uint64).view(np.uint8)
        kernarg[96:104] = np.array([rows.shape[1] * 4, (len(plan[5]) * 4 - gen.TILE_HEADER) // gen.image_bytes()], dtype=np.uint32).view(np.uint8)
        kernarg[104:112] = np.array(fused[2:], dtype=np.uint64).view(np.uint8)
    where = memory.add(kernarg)
    kernel = _kernel(gen, depth, six, rows is not None)
    for block in range(blocks):
        lds = _Lds(gen.lds_bytes(depth, six, rows is not None), rng)
        waves = [_Wave(kernel, memory, lds, where, block, w) for w in range(16)]
        running = list(range(16))
        while running:
            ended = []
            for w in rng.permutation(running):
                if waves[w].run():
                    ended.append(w)
            assert not ended or len(ended) in (12, len(running))
            running = [w for w in running if w not in ended]
    return out


# trees, buckets, depths, bins up to, share of one-hot levels, skewed buckets, documents
CASES = [
    (1, 3, [8], 127, 0.0, False, 1),
    (31, 700, [8], 127, 0.02, False, 300),
    (97, 1024, [8], 63, 0.05, False, 256),
    (200, 600, [1, 4, 6, 7, 8], 127, 0.1, True, 200),
    (130, 900, [0, 7, 8], 63, 0.0, True, 511),
    (161, 640, [4, 5, 6], 127, 0.02, False, 256),
    (64, 1000, [6], 63, 0.3, False, 255),
    (33, 20, [2, 6], 63, 0.0, True, 256),
]


@pytest.mark.parametrize("case", CASES, ids=[str(c[:3]) for c in CASES])
def test_kernel_on_planned_tables(planner, tmp_path, case):
    tree_count, buckets, depths, limit, one_hot, skew, docs = case
    gen = _generator()
    rng = np.random.default_rng(tree_count * 1000 + buckets)
    depth = 6 if max(depths) <= 6 else 8
    trees = _model(rng, tree_count, buckets, depths, limit, one_hot, skew)
    bins = rng.integers(0, limit + 1, size=((docs + 255) // 256 * 256, buckets)).astype(np.uint8)
    for six in (False, True) if limit <= 63 else (False,):
        plan = _plan(planner, str(tmp_path / "model.txt"), trees, buckets, depth, six)
        assert plan is not None
        got = _run(gen, plan, bins, docs, buckets, depth, six, 0.5, 0.25, rng)
        np.testing.assert_array_equal(got, _expected(trees, bins)[:docs] * 0.5 + 0.25)


# trees, columns, one-hot columns, depths, borders up to, documents
FUSED_CASES = [
    (40, 70, 0, [8], 60, 300),          # a last tile of two pieces, and documents behind the last row
    (33, 1016, 16, [7, 8], 60, 256),    # sixteen tiles, one-hot columns in the last ones
    (48, 200, 21, [6], 63, 41),         # more one-hot columns in a tile than waves
    (35, 130, 5, [8], 127, 257),        # seven bits
    (16, 66, 3, [5, 6], 120, 1),
]


@pytest.mark.parametrize("case", FUSED_CASES, ids=[str(c[:3]) for c in FUSED_CASES])
def test_fused_kernel_on_rows(planner, tmp_path, case):
    """A column in three is not used, some pieces are not: a piece that would leave the row is moved back over its neighbour. The
    documents hold borders, values next to them, infinities, NaN, denormals and hashes of no category."""
    tree_count, columns, one_hot, depths, limit, docs = case
    gen = _generator()
    rng = np.random.default_rng(tree_count * 1000 + columns)
    used = np.flatnonzero(rng.random(columns) < (0.97 if columns > 900 else 0.7))
    is_hot = np.zeros(columns, dtype=bool)
    is_hot[rng.permutation(used[used > columns // 2] if columns > 900 else used)[:one_hot]] = True
    pieces, column_of, covered = [], {}, -1
    for c in used:
        if c > covered:
            start = min(c & ~3, columns - 4)
            pieces.append(start)
            covered = start + 3
        column_of[c] = (len(pieces) - 1) // 16 * 64 + (len(pieces) - 1) % 16 * 4 + c - pieces[-1]
    pieces += [0] * (-len(pieces) % 16)
    assert len(pieces) <= 256
    rows = rng.normal(size=(docs, columns)).astype(np.float32)
    table = [(0, 0, 0, [])] * (4 * len(pieces))
    bins = np.zeros(((docs + 255) // 256 * 256, len(used)), dtype=np.uint8)
    six = limit <= 63
    count = np.zeros(len(used), dtype=int)
    for b, c in enumerate(used):
        n = count[b] = int(rng.integers(1, limit + 1))
        if is_hot[c]:
            n = count[b] = min(n, 20)
            values = rng.choice(2**31, size=n, replace=False).astype(np.uint32)
            hashes = np.append(values, np.uint32(12345))[rng.integers(0, n + 1, size=docs)]
            rows[:, c] = hashes.view(np.float32)
            bins[:docs, b] = ((hashes[:, None] == values) * np.arange(1, n + 1)).max(axis=1)
            table[column_of[c]] = (1, 1, 4 * c, values)
            continue
        # (normal values of a float's every size in a column or two, else at most fifteen borders may share a cell)
        borders = np.unique(rng.normal(size=n).astype(np.float32)) if c % 3 else np.linspace(-1, 1, n).astype(np.float32)
        if c % 7 == 0:
            borders = np.float32([-3e38, 1e-40, 1.0, 3e38])
        count[b] = len(borders)
        special = np.concatenate([borders, np.nextafter(borders, np.float32(9)), [np.inf, -np.inf, np.nan, 1e-40, 3e38, -3e38]]).astype(np.float32)
        at = rng.random(docs) < 0.3
        rows[at, c] = rng.choice(special, size=at.sum())
        with np.errstate(invalid="ignore"):
            bins[:docs, b] = (rows[:, c:c + 1] > borders).sum(axis=1)
        table[column_of[c]] = (1, 0, 0, borders.view(np.uint32))
    depth = 6 if max(depths) <= 6 else 8
    trees = []
    for t in range(tree_count):
        levels = [(int(b), int(rng.integers(1, count[b] + 1)), bool(is_hot[used[b]]))
                  for b in rng.integers(0, len(used), size=int(rng.choice(depths)))]
        trees.append((levels, rng.normal(size=1 << len(levels))))
    tiles = ([column_of[c] for c in used], [4 * p for p in pieces], table)
    plan = _plan(planner, str(tmp_path / "model.txt"), trees, len(used), depth, six, tiles)
    assert plan is not None and len(plan) == 7
    got = _run(gen, plan, bins, docs, len(used), depth, six, 0.5, 0.25, rng, rows=rows)
    np.testing.assert_array_equal(got, _expected(trees, bins)[:docs] * 0.5 + 0.25)


@pytest.mark.parametrize("docs,six,depths", [(256, True, [8]), (255, False, [1, 5, 7, 8])])
def test_kernel_on_folded_leaf_rows(planner, tmp_path, monkeypatch, docs, six, depths):
    """The form that is built for depth 8: leaf l of a row stands at l ^ (l >> 1)."""
    import functools

    def bitop3(wave, args):
        last, table = args[3].split()
        x, y, z = wave.vector(args[1], True), wave.vector(args[2]), wave.vector(last)
        assert table == "bitop3:0x6a"
        wave._set(args, (x & y) ^ z)
    monkeypatch.setattr(_Wave, "op_v_bitop3_b32", bitop3, raising=False)
    gen = _generator()
    assert gen.folds_leaves(8) and not gen.folds_leaves(6)
    monkeypatch.setattr(gen, "gen_kernel", functools.partial(gen.gen_kernel, folded=True))
    rng = np.random.default_rng(docs)
    trees = _model(rng, 70, 600, depths, 63 if six else 127, 0.0)
    bins = rng.integers(0, 64 if six else 128, size=(256, 600)).astype(np.uint8)
    plan = list(_plan(planner, str(tmp_path / "model.txt"), trees, 600, 8, six))
    place = np.arange(256) ^ (np.arange(256) >> 1)
    folded = np.empty((plan[4].size // 256, 256))
    folded[:, place] = plan[4].reshape(-1, 256)
    plan[4] = folded.reshape(-1)
    got = _run(gen, plan, bins, docs, 600, 8, six, 0.5, 0.25, rng)
    np.testing.assert_array_equal(got, _expected(trees, bins)[:docs] * 0.5 + 0.25)


def test_plan_refuses_more_buckets_than_registers(planner, tmp_path):
    rng = np.random.default_rng(5)
    trees = [([(b, 1, False)], rng.normal(size=2)) for b in range(1025)]
    assert _plan(planner, str(tmp_path / "model.txt"), trees, 1025, 8, False) is None
    assert _plan(planner, str(tmp_path / "model.txt"), trees[:1024], 1025, 8, False) is not None


def test_plan_of_a_large_model(planner, tmp_path):
    """5000 trees over 1016 buckets: every group is compared once, about one per wave and step, and the waves share the levels evenly."""
    rng = np.random.default_rng(11)
    trees = _model(rng, 5000, 1016, [8], 60, 0.016)
    rounds, wave_table, records, extra_rows, leaves = _plan(planner, str(tmp_path / "model.txt"), trees, 1016, 8, True)
    rows = records.reshape(rounds + 1, 16, 96)[:rounds, :, :64].reshape(rounds, 16, 4, 16)
    skipped = (rows[..., 2] >> 29 & 1).sum(axis=(0, 2))
    extra = np.diff(np.append(wave_table.reshape(16, 80)[:, 64] // 64, len(extra_rows) // 16))
    groups = 4 * rounds - skipped + extra
    levels = sum(len(t[0]) for t in trees)
    assert groups.max() <= 1.02 * groups.mean() and levels <= groups.sum() * 8 < levels + 16 * 8
    late = extra - wave_table.reshape(16, 80)[:, 65]           # more than one group in a step
    assert (late >= 0).all() and late.sum() < 0.03 * groups.sum()


@pytest.mark.parametrize("trees,share,least,most", [
    (2000, 0.0, 1.0, 1.4), (2000, 0.1, 1.5, 2.1), (2000, 0.3, 4.0, 5.2),
    (60, 0.0, 0.75, 1.8), (60, 0.5, 5.0, 9.0),          # one round: all groups are compared before it, none behind its last step
])
def test_plan_says_how_much_longer_the_busiest_waves_compare(planner, tmp_path, trees, share, least, most):
    """A bucket's levels are all compared by the wave that holds it: with `share` of them on one bucket, 16 * share of a wave's part."""
    rng = np.random.default_rng(3)
    model = [([(0 if rng.random() < share else int(rng.integers(0, 1000)), 60, False) for _ in range(8)], np.zeros(256))
             for _ in range(trees)]
    path = str(tmp_path / "model.txt")
    _plan(planner, path, model, 1000, 8, True)
    steps, compared = map(int, subprocess.check_output([planner, path, "steps"], text=True).split())
    assert least <= compared / steps <= most
