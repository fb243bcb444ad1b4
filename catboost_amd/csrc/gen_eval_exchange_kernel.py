"""Writes the gfx950 assembly of the exchange kernels: one-dimensional oblivious models of depth <= 8 whose bins of a 256-document
block are too many for one wave's registers (up to 1024 buckets) but fit the registers of a workgroup's sixteen waves.

  * wave w keeps 64 buckets of the block, one register each (four documents per lane as in the register kernels), so a
    level costs no read of its bins. It compares the levels that look at its buckets, whichever tree they belong to, and
    packs the results of DEPTH levels (a *group*) into a dword of four documents, one bit each: register index through M0, an
    add whose carry is the result, a shift and a bit-field insert;
  * a group's dword goes to an LDS slot of 256 bytes; the wave that sums a tree reads the DEPTH slots its row names and
    takes the bit of position p from the p-th: the host has placed the levels so that no two of a tree or of a
    group share a position (exchange_plan.h), so seven bit-field inserts make the leaf indexes. A position that the
    tree has no level for holds some other bit; the tree's leaf values are repeated there;
  * tree t of pair p = t / 2 is summed by wave p % 16, in order, and the sixteen sums are added in the order of the waves: the
    pair-tile kernel's sums, bit for bit;
  * a *step* is one tree per wave, a *round* four steps and a barrier. Groups are compared one per step (rows can skip one
    or name more) at least a round before a tree looks at them;
  * every wait of a step is for requests made a step earlier: the dwords of the next tree are read, and the rows of the
    next group and the tree after next requested, right behind the step's one wait for LDS and scalar loads, the leaf
    values gathered before the step's group is compared, and added behind the next step's wait;
  * a tree's leaf values go from global memory to the wave's own LDS region (three regions per wave, two steps ahead).

What bounds it: LDS. Per tree and 256 documents 36 vector and 26 scalar instructions, and of the 100 cycles (at the 2.34 GHz it runs at, fused
form) that a step of sixteen waves takes for each 56 of reads (by its counters: four gathers and nine dwords, the bins' tables; 23 of them bank
conflicts, 28 before the leaf rows were folded) and 32 for the 2 KB of leaf values, which come in at 64 bytes per clock; the pair-tile kernel, in which only
128 documents share a copy of the leaf values and every level reads its bins, issues 82 vector instructions. Over bins from memory and before
the fold (84 cycles of 2.4 GHz), 262 144 documents x 5000 trees x 1016 buckets 0.70 ms; with half of the leaf values' copies left out 0.60, without the gathers 0.60, without reading the groups' dwords
0.59, without the barriers 0.68, without loading rows 0.69. Tried: every request in the step that waits for it 0.77, slots
addressed by vector registers (nine more vector instructions) 0.72, leaf values through registers and ds_write_b128 0.78, one
tree in four gathered from global memory 0.70. Some 13 us per workgroup go to its start (the bins, the first groups) and end.

Fused variants ("cbamd_fused_exchange_...") take the documents' rows and make the bins themselves, tile by tile: a tile is sixteen
*pieces* of four neighbouring columns (16 bytes of a row). A lane loads a piece of its four documents (sixteen lanes a row's
pieces, so a load reads whole stretches of four rows), finds the bins as the other fused kernels do - cell of a grid of
256 (six-bit form 512), table of search starts, a branch-free search of 1 to 4 steps - with its columns' borders and start tables in LDS, and
writes a dword of four documents' bins per column to a buffer [column][lane] in LDS, from which every wave takes the four of its
64 buckets that are in this tile. A tile's tables come straight into LDS while the tile before is searched, its rows
likewise into registers. One-hot columns are made behind that, by a wave per column. The phase takes some 55 us per workgroup of
1016 columns: with all CUs in it at once 43 us are the rows' way from HBM (6.2 TB/s), with rows that sit in L2 it takes 45, at 43 %
of the vector issue (12 instructions per value and search of two steps) and 36 % of LDS; the binarize launch and reading its bins took
70 us of each workgroup's documents. Before the pieces' tables stood in different banks it took 80 us with few borders per column;
four searches side by side instead of eight, a grid of 256 cells and a cell in five instructions instead of three: 5 to 8 us more each.
1M documents over 1016 features, whole call, two launches -> fused: 500 trees of depth 8 1.53 -> 1.26 ms, 5000 3.77 -> 3.51.

Kernel arguments (80 bytes, fused 112):
   0 bins const uint32* [docBlock][bucketCount][64]      8 wave table const uint32* [16][80]
  16 records const uint32* [rounds + 1][16][96]         24 extra group rows const uint32*
  32 leaves const double* [rounds + 1][16][4][1 << DEPTH]   40 out double* [docCount]
  48 bias const double*                                 56 scale double
  64 docCount uint32   68 rounds uint32 (>= 1)   72 bytes of a document block's bins uint32
  fused: the bins are not there, the wave table's offsets are byte offsets of columns in the buffer
  80 rows const float*   88 tile table const uint32* (TILE_HEADER bytes, then an image per tile)
  96 row stride in bytes uint32   100 tiles uint32 (1 .. 16)   104 one-hot columns const uint32*
grid = document blocks, 1024 threads; LDS: the slots, then sixteen times three leaf regions; at the end the partial sums.
"""

import struct

WAVES = 16
WAVE_BUCKETS = 64
ROUND_STEPS = 4
SLOTS = 224
REGIONS = 3
WAVE_TABLE_BYTES = 320
GROUP_BYTES = 64
TREE_ROW_BYTES = 32
EARLY_ROWS = 3            # rows of the groups before the first step that are fetched together
RECORD_BYTES = ROUND_STEPS * (GROUP_BYTES + TREE_ROW_BYTES)
SKIP_FLAG = 0x20000000  # the lowest of a group row's flags

# the fused kernels' binarize phase
TILES = 16
TILE_COLUMNS = 64
COLUMN_BYTES = 260         # of the buffer: 64 dwords and one more, so that a tile's columns start in different banks
OFFSETS_AT = 256           # behind the tiles' infos (16 bytes: search steps, one-hot columns, byte offset of their list): per tile the
                           # byte offsets of its pieces in a row
TILE_HEADER = OFFSETS_AT + TILES * 64
PARAMETERS_BYTES = 768     # of an image: per piece 48 bytes, four scale, four bias, the next tile's piece, three spare dwords
TABLE_BYTES = 768          # of a column in an image: its borders, then the search starts of its grid's cells
ONE_HOT_BYTES = 64         # record of a one-hot column: byte offset in a row, offset in the buffer, records of values; then those
MAX_STEPS = 4
BUFFERS = [0, TILE_COLUMNS * COLUMN_BYTES]
IMAGES_AT = 33 * 1024

SHAPES = [(depth, six, fused) for fused in (False, True) for depth in (8, 6) for six in (False, True)]


def border_bytes(six):
    return 256 if six else 512


def grid_cells(six):
    return TABLE_BYTES - border_bytes(six)


# From one piece's tables to the next one's: sixteen bytes more than their size, so that pieces whose lanes look at the same place of
# their tables (few borders, values that agree) look at different banks.
PIECE_BYTES = 4 * TABLE_BYTES + 16


def image_bytes():
    return TILE_COLUMNS // 4 * PIECE_BYTES + PARAMETERS_BYTES


def folds_leaves(depth):
    """Whether a kernel's leaf rows are folded (PlaceLeavesKernel: leaf l stands at l ^ (l >> 1)): the leaves that share an LDS bank then
    differ in more levels, and fewer of a bank's rows are wanted at a time. 2M documents x 5000 trees of depth 8 x 1016 buckets 6707 ->
    6582 us, for two vector instructions; with 64 leaves, which have two rows to a bank and not eight, 2960 -> 2990 (1M, depth 6)."""
    return depth == 8


def kernel_name(depth, six, fused=False):
    return "cbamd_%s_exchange_d%d%s" % ("fused" if fused else "eval", depth, "_s" if six else "")


def lds_bytes(depth, six=False, fused=False):
    walk = SLOTS * 256 + WAVES * REGIONS * (8 << depth)
    return max(walk, IMAGES_AT + 2 * image_bytes()) if fused else walk


def gen_kernel(depth, six, fused=False, folded=False):
    """folded: the leaf rows are (folds_leaves)."""
    name = kernel_name(depth, six, fused)
    leaf_bytes = 8 << depth
    round_leaf_bytes = WAVES * ROUND_STEPS * leaf_bytes
    round_record_bytes = WAVES * RECORD_BYTES
    pieces = max(1, leaf_bytes // 1024)
    first_bit = 8 - depth
    assert SLOTS * 256 >= WAVES * 256 * 8      # the partial sums take the slots' place

    # scalar registers
    groups = [32, 48]                          # the rows of the groups of even and odd steps
    tree_rows = [80, 88]                       # the rows of even and odd steps' trees
    masks = [8, 9, 10, 11, 28, 29, 30, 31]     # 0x01010101 << place
    high_bits, pair_bits = 96, 97
    regions = [98, 99, 100]                    # LDS addresses of the wave's leaf regions
    # vector registers: v0 thread, v1 lane * 4, v2 lane * 16, v3 .. v5 group
    dwords = [6, 40]                           # the dwords of even and odd steps' trees
    ga0, lv0, ac0, sc0, b0 = 14, 18, 26, 34, 64
    vgprs = b0 + WAVE_BUCKETS

    o = []
    e = o.append

    def load_extra(regs):
        """The wave's next extra group row."""
        e("  s_load_dwordx16 s[%d:%d], s[12:13], 0x0" % (regs, regs + 15))
        e("  s_add_u32 s12, s12, %d" % GROUP_BYTES)
        e("  s_addc_u32 s13, s13, 0")

    def compare_levels(group, xors):
        # the first level needs no masking with eight levels: what it leaves below its bit moves out of the byte or is
        # overwritten (six levels: two bits stay, the tree's wave masks them)
        def level(d, to):
            e("  s_set_gpr_idx_%s" % ("on s%d, 0x1" % group if d == 0 else "idx s%d" % (group + 2 * d)))
            if xors:
                e("  s_bfe_u32 s4, s%d, 0x80008" % (group + 2 * d))
                e("  s_mul_i32 s4, s4, 0x01010101")
                e("  v_xor_b32_e64 v%d, v%d, s4" % (to, b0))
                e("  v_add_u32_e32 v%d, s%d, v%d" % (to, group + 2 * d + 1, to))
            else:
                e("  v_add_u32_e64 v%d, v%d, s%d" % (to, b0, group + 2 * d + 1))
        if six:
            for pair in range(depth // 2):
                level(2 * pair, 4)
                level(2 * pair + 1, 3 if pair == 0 else 5)
                if pair == 0:
                    e("  v_bfi_b32 v3, s%d, v3, v4" % high_bits)
                else:
                    e("  v_bfi_b32 v4, s%d, v5, v4" % high_bits)
                    e("  v_lshrrev_b32_e32 v3, 2, v3")
                    e("  v_bfi_b32 v3, s%d, v4, v3" % pair_bits)
        else:
            for d in range(depth):
                level(d, 3 if d == 0 else 4)
                if d > 0:
                    e("  v_lshrrev_b32_e32 v3, 1, v3")
                    e("  v_bfi_b32 v3, s%d, v4, v3" % high_bits)
        e("  s_set_gpr_idx_off")
        # its dword into its slot
        e("  s_lshr_b32 m0, s%d, 16" % group)
        e("  s_nop 0")                          # a wait state between M0 and the write
        e("  ds_write_addtid_b32 v3")

    out_of_line = []

    def compare_group(group, label):
        """The group whose row is in `group`, and those that follow it in the wave's extra rows."""
        e("  s_cmp_gt_u32 s%d, 0x%x" % (group + 2, SKIP_FLAG - 1))
        e("  s_cbranch_scc1 %s_flags" % label)
        compare_levels(group, False)
        e("%s_compared:" % label)

        def by_flags():
            e("%s_flags:" % label)
            e("  s_bitcmp1_b32 s%d, 29" % (group + 2))
            e("  s_cbranch_scc1 %s_compared" % label)
            e("  s_bitcmp1_b32 s%d, 31" % (group + 2))
            e("  s_cbranch_scc1 %s_xor" % label)
            compare_levels(group, False)
            e("%s_next:" % label)
            e("  s_bitcmp1_b32 s%d, 30" % (group + 2))
            e("  s_cbranch_scc0 %s_compared" % label)
            load_extra(group)
            e("  s_waitcnt lgkmcnt(0)")
            e("  s_branch %s_flags" % label)
            e("%s_xor:" % label)
            compare_levels(group, True)
            e("  s_branch %s_next" % label)
        out_of_line.append(by_flags)

    def fetch_leaves(region, second):
        """Leaf values at s[16:17], or behind those, into an LDS region."""
        offset = leaf_bytes if second else 0    # moves the source and the destination
        if second:
            e("  s_sub_u32 m0, s%d, 0x%x" % (region, offset))
        else:
            e("  s_mov_b32 m0, s%d" % region)
        if leaf_bytes < 1024:
            e("  s_mov_b32 exec_hi, 0")         # 32 lanes of 16 bytes
        else:
            e("  s_nop 0")                      # a wait state between M0 and the copy
        for piece in range(pieces):
            at = offset + piece * 1024
            e("  global_load_lds_dwordx4 v2, s[16:17]%s" % (" offset:%d" % at if at else ""))
        if leaf_bytes < 1024:
            e("  s_mov_b32 exec_hi, -1")

    def advance(pointer, by):
        e("  s_add_u32 s%d, s%d, 0x%x" % (pointer, pointer, by))
        e("  s_addc_u32 s%d, s%d, 0" % (pointer + 1, pointer + 1))

    # rows of a step of this round or the next one's first two (s[14:15]: the wave's record of this round)
    def load_group_row(step):
        at = step // ROUND_STEPS * round_record_bytes + step % ROUND_STEPS * GROUP_BYTES
        regs = groups[step % 2]
        e("  s_load_dwordx16 s[%d:%d], s[14:15], 0x%x" % (regs, regs + 15, at))

    def load_tree_row(step):
        at = step // ROUND_STEPS * round_record_bytes + ROUND_STEPS * GROUP_BYTES + step % ROUND_STEPS * TREE_ROW_BYTES
        regs = tree_rows[step % 2]
        e("  s_load_dwordx8 s[%d:%d], s[14:15], 0x%x" % (regs, regs + 7, at))

    def read_dwords(step, between):
        """The dwords that the tree's row names (their slots' addresses go through M0), with independent instructions in the wait
        state between M0 and the read."""
        for d in range(depth):
            e("  s_mov_b32 m0, s%d" % (tree_rows[step % 2] + d))
            e(between.pop(0) if between else "  s_nop 0")
            e("  ds_read_addtid_b32 v%d" % (dwords[step % 2] + d))
        for line in between:
            e(line)

    def sums():
        """The last tree's values are added."""
        return ["  v_add_f64 v[%d:%d], v[%d:%d], v[%d:%d]" % (ac0 + 2 * j, ac0 + 2 * j + 1, ac0 + 2 * j, ac0 + 2 * j + 1,
                                                              lv0 + 2 * j, lv0 + 2 * j + 1) for j in range(4)]

    def leaf_indexes(dw0):
        """A tree's leaf indexes, a byte per document, into v3."""
        out = ["  v_bfi_b32 v3, s%d, v%d, v%d" % (masks[first_bit], dw0, dw0 + 1)]
        out += ["  v_bfi_b32 v3, s%d, v%d, v3" % (masks[first_bit + d], dw0 + d) for d in range(2, depth)]
        if depth < 8:
            out.append("  v_and_b32_e32 v3, 0x%x, v3" % (((0xff << first_bit) & 0xff) * 0x01010101))
        if folded:
            out.append("  v_lshrrev_b32_e32 v38, 1, v3")
            out.append("  v_bitop3_b32 v3, v38, v39, v3 bitop3:0x6a")
        return out

    def step(number):
        """Step i of a round; `number` counts the steps of a turn of the loop."""
        i = number % ROUND_STEPS
        here = regions[number % REGIONS]
        # this tree's dwords, the last tree's leaf values, the next rows, the last group in its slot: all requested a step ago
        e("  s_waitcnt lgkmcnt(0)")
        load_tree_row(i + 2)
        load_group_row(i + 1)
        if i == ROUND_STEPS - 1:
            e("  s_barrier")
        read_dwords(i + 1, sums() + leaf_indexes(dwords[i % 2]))
        for j in range(4):
            e("  v_dot4_u32_u8 v%d, v3, v%d, s%d" % (ga0 + j, sc0 + j, here))
        e("  s_waitcnt vmcnt(%d)" % pieces)     # this tree's leaf values; the next one's may still be under way
        for j in range(4):
            e("  ds_read_b64 v[%d:%d], v%d" % (lv0 + 2 * j, lv0 + 2 * j + 1, ga0 + j))
        # the last tree's values have been gathered: its region takes the ones two steps ahead
        if i % 2 == 0:
            advance(16, 2 * leaf_bytes if i == 0 else round_leaf_bytes - 2 * leaf_bytes)
        fetch_leaves(regions[(number + 2) % REGIONS], i % 2 == 1)
        compare_group(groups[i % 2], "%s_t%d" % (name, number))

    def binarize_tiles():
        """The binarize phase: the wave's bins from the documents' rows. Vector registers below the bins but v1 are free,
        scalar registers from 26 on."""
        two, tile, following, left, table, wave_lists = 26, 27, 28, 29, 30, 32
        stride, tiles, one_hot, register, last = 34, 35, 36, 38, 39
        infos, lists = [64, 68], [72, 76]
        highest_cell = 101
        rows_base, rows_there = [80, 82, 84, 86], [88, 90, 92, 94]  # per document of a lane: its rows' base, the lanes that have one
        table_of_float, two_to_23, tables = 0, 2, 3      # tables - the bits of 2^23; 2^23; LDS address of the piece's tables
        scale, bias, offset, out = 4, 8, 12, 12
        values, place, probe = [16, 32], 48, 56
        image = image_bytes()
        per_wave = image // WAVES // 1024 * 1024
        copies = per_wave // 1024 + 1
        assert image == WAVES * per_wave + 1024
        assert IMAGES_AT >= BUFFERS[1] + TILE_COLUMNS * COLUMN_BYTES and IMAGES_AT % 1024 == image % 1024 == 0
        # byte of a position's dword that belongs to the piece and not to the bin: (piece * PIECE_BYTES / 4) % 256 = 4 * piece
        assert PIECE_BYTES // 4 % 256 == 4 and 4 * (TILE_COLUMNS // 4 - 1) + border_bytes(six) // 4 < 256

        def copy_image(x):
            """The following tile's image: the wave's share of it, the last 1 KB (with the parameters) by every wave alike."""
            e("  v_lshlrev_b32_e32 v%d, 2, v1" % probe)
            e("  s_mul_i32 s4, s3, 0x%x" % per_wave)
            e("  s_mul_i32 s5, s%d, 0x%x" % (following, image))
            e("  s_add_u32 s5, s5, 0x%x" % TILE_HEADER)
            e("  s_add_u32 s6, s4, s5")
            e("  s_add_u32 s6, s%d, s6" % table)
            e("  s_addc_u32 s7, s%d, 0" % (table + 1))
            e("  s_add_u32 m0, s4, 0x%x" % (IMAGES_AT + x * image))
            e("  s_nop 0")
            for piece in range(copies - 1):
                e("  global_load_lds_dwordx4 v%d, s[6:7]%s" % (probe, " offset:%d" % (piece * 1024) if piece else ""))
            e("  s_add_u32 s5, s5, 0x%x" % (image - 1024))
            e("  s_add_u32 s6, s%d, s5" % table)
            e("  s_addc_u32 s7, s%d, 0" % (table + 1))
            e("  s_mov_b32 m0, 0x%x" % (IMAGES_AT + (x + 1) * image - 1024))
            e("  s_nop 0")
            e("  global_load_lds_dwordx4 v%d, s[6:7]" % probe)

        def load_values(x):
            """(A lane without a document keeps what its registers hold.)"""
            e("  v_lshrrev_b32_e32 v%d, 6, v1" % probe)
            e("  s_lshl_b32 s4, s3, 2")
            e("  v_add_u32_e32 v%d, s4, v%d" % (probe, probe))
            e("  v_mul_lo_u32 v%d, v%d, s%d" % (probe, probe, stride))
            e("  v_add_u32_e32 v%d, v%d, v%d" % (probe, probe, offset))
            for j in range(4):
                e("  s_mov_b64 exec, s[%d:%d]" % (rows_there[j], rows_there[j] + 1))
                e("  global_load_dwordx4 v[%d:%d], v%d, s[%d:%d]" % (values[x] + 4 * j, values[x] + 4 * j + 3, probe, rows_base[j], rows_base[j] + 1))
            e("  s_mov_b64 exec, -1")

        def load_infos(x):
            """The following tile's."""
            e("  s_lshl_b32 s4, s%d, 4" % following)
            for regs, base in ((infos[x], table), (lists[x], wave_lists)):
                e("  s_add_u32 s6, s%d, s4" % base)
                e("  s_addc_u32 s7, s%d, 0" % (base + 1))
                e("  s_load_dwordx4 s[%d:%d], s[6:7], 0x0" % (regs, regs + 3))

        def next_tile():
            """`tile` and `following` move on, round the end."""
            e("  s_mov_b32 s%d, s%d" % (tile, following))
            e("  s_add_u32 s%d, s%d, 1" % (following, following))
            e("  s_cmp_eq_u32 s%d, s%d" % (following, tiles))
            e("  s_cselect_b32 s%d, 0, s%d" % (following, following))

        def search(label, x, j):
            """The bins of the lane's documents j and j + 1 in its four columns, eight searches side by side, into bytes j and
            j + 1 of the columns' dwords."""
            value = values[x] + 4 * j

            def step(number):
                size = 4 << (number - 1)
                for k in range(8):
                    e("  ds_read_b32 v%d, v%d offset:%d" % (probe + k, place + k, k % 4 * TABLE_BYTES + size - 4))
                e("  s_waitcnt lgkmcnt(0)")
                for k in range(8):
                    e("  v_cmp_lt_f32_e32 vcc, v%d, v%d" % (probe + k, value + k))
                    e("  v_cndmask_b32_e64 v%d, 0, %d, vcc" % (probe + k, size))
                    e("  v_add_u32_e32 v%d, v%d, v%d" % (place + k, place + k, probe + k))
            for k in range(8):
                c = k % 4
                # the value's cell, 0 .. highest_cell, in the low bits of 2^23 + cell; NaN (and -inf) in the first one
                e("  v_fma_f32 v%d, v%d, v%d, v%d clamp" % (probe + k, value + k, scale + c, bias + c))
                e("  v_fma_f32 v%d, v%d, s%d, v%d" % (probe + k, probe + k, highest_cell, two_to_23))
                e("  v_add_u32_e32 v%d, v%d, v%d" % (probe + k, probe + k, table_of_float))
                e("  ds_read_u8 v%d, v%d offset:%d" % (place + k, probe + k, c * TABLE_BYTES + border_bytes(six)))
            e("  s_waitcnt lgkmcnt(0)")
            for k in range(8):
                if six:
                    e("  v_add_u32_e32 v%d, v%d, v%d" % (place + k, place + k, tables))
                else:
                    e("  v_lshl_add_u32 v%d, v%d, 2, v%d" % (place + k, place + k, tables))
            for number in range(MAX_STEPS, 1, -1):
                e("  s_cmp_lt_u32 s%d, %d" % (infos[x], number))
                e("  s_cbranch_scc1 %s_%d_below%d" % (label, j, number))
                step(number)
                e("%s_%d_below%d:" % (label, j, number))
            step(1)
            for k in range(8):
                # bits 2 .. 9: the bin and what the place of the piece's tables adds to it
                e("  v_lshrrev_b32_sdwa v%d, s%d, v%d dst_sel:BYTE_%d dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD"
                  % (out + k % 4, two, place + k, j + k // 4))

        def one_hot_columns(label, x):
            """A wave per one-hot column of the tile (column k of them by wave k % 16), behind the other columns."""
            e("%s_hot:" % label)
            e("  s_waitcnt lgkmcnt(0)")
            e("  s_barrier")                       # the dwords of these columns that the lanes have written are overwritten
            e("  s_mov_b32 s40, s3")
            e("  s_lshl_b32 s4, s3, 2")
            e("  s_add_u32 s6, s%d, s%d" % (one_hot, infos[x] + 2))
            e("  s_addc_u32 s7, s%d, 0" % (one_hot + 1))
            e("  s_add_u32 s6, s6, s4")
            e("  s_addc_u32 s7, s7, 0")
            e("%s_hot_next:" % label)
            e("  s_cmp_ge_u32 s40, s%d" % (infos[x] + 1))
            e("  s_cbranch_scc1 %s_hot_done" % label)
            e("  s_load_dword s41, s[6:7], 0x0")   # byte offset of the column's record
            e("  s_waitcnt lgkmcnt(0)")
            e("  s_add_u32 s42, s%d, s41" % one_hot)
            e("  s_addc_u32 s43, s%d, 0" % (one_hot + 1))
            e("  s_load_dwordx4 s[44:47], s[42:43], 0x0")    # offset in a row, offset in the buffer, records of eight values
            e("  s_waitcnt lgkmcnt(0)")
            # all documents of the block, lane l's are l, l + 64 ..; the tile's own values are no longer needed
            for j in range(4):
                e("  v_lshrrev_b32_e32 v%d, 2, v1" % (place + j))
                e("  v_add_u32_e32 v%d, %d, v%d" % (place + j, 64 * j, place + j))
                e("  v_min_u32_e32 v%d, s%d, v%d" % (place + j, last, place + j))
                e("  v_mul_lo_u32 v%d, v%d, s%d" % (place + j, place + j, stride))
                e("  v_add_u32_e32 v%d, s44, v%d" % (place + j, place + j))
            for j in range(4):
                e("  global_load_dword v%d, v%d, s[%d:%d]" % (values[x] + j, place + j, rows_base[0], rows_base[0] + 1))
            for j in range(4):
                e("  v_mov_b32_e32 v%d, 0" % (probe + j))
            e("  s_waitcnt vmcnt(0)")
            e("%s_hot_values:" % label)
            e("  s_add_u32 s42, s42, %d" % ONE_HOT_BYTES)
            e("  s_addc_u32 s43, s43, 0")
            e("  s_load_dwordx16 s[48:63], s[42:43], 0x0")   # eight times (value, bin)
            e("  s_waitcnt lgkmcnt(0)")
            for i in range(8):
                e("  v_mov_b32_e32 v%d, s%d" % (place, 49 + 2 * i))
                for j in range(4):
                    e("  v_cmp_eq_u32_e32 vcc, s%d, v%d" % (48 + 2 * i, values[x] + j))
                    e("  v_cndmask_b32_e32 v%d, v%d, v%d, vcc" % (probe + j, probe + j, place))
            e("  s_sub_u32 s46, s46, 1")
            e("  s_cmp_lg_u32 s46, 0")
            e("  s_cbranch_scc1 %s_hot_values" % label)
            for j in range(1, 4):
                e("  v_lshl_or_b32 v%d, v%d, %d, v%d" % (probe, probe + j, 8 * j, probe))
            e("  s_mov_b32 m0, s45")
            e("  s_nop 0")
            e("  ds_write_addtid_b32 v%d offset:%d" % (probe, BUFFERS[x]))
            e("  s_add_u32 s40, s40, %d" % WAVES)
            e("  s_add_u32 s6, s6, %d" % (4 * WAVES))
            e("  s_addc_u32 s7, s7, 0")
            e("  s_branch %s_hot_next" % label)
            e("%s_hot_done:" % label)
            e("  s_branch %s_hot_back" % label)

        def read_bins(x):
            """The wave's four columns of a tile, behind its barrier."""
            for i in range(4):
                e("  s_mov_b32 m0, s%d" % (lists[x] + i))
                e("  s_nop 0")
                e("  ds_read_addtid_b32 v%d offset:%d" % (place + i, BUFFERS[x]))

        def take_bins():
            """... into their registers (before the first tile: of no tile, into the first one's registers, which are written again)."""
            e("  s_set_gpr_idx_on s%d, 0x8" % register)
            for i in range(4):
                e("  v_mov_b32_e32 v%d, v%d" % (b0 + i, place + i))
            e("  s_set_gpr_idx_off")
            e("  s_lshl_b32 s%d, s%d, 2" % (register, tile))

        def lane_piece(piece, document):
            """The lane's piece, and its first document of the block: 4 * wave + lane / 16."""
            e("  v_lshrrev_b32_e32 v%d, 6, v1" % document)
            e("  s_lshl_b32 s4, s3, 2")
            e("  v_add_u32_e32 v%d, s4, v%d" % (document, document))
            e("  v_bfe_u32 v%d, v1, 2, 4" % piece)

        e("  s_load_dwordx8 s[40:47], s[0:1], 0x50")    # rows, tile table, stride, tiles, one-hot columns
        e("  s_waitcnt lgkmcnt(0)")
        e("  s_mov_b64 s[%d:%d], s[42:43]" % (table, table + 1))
        e("  s_mov_b64 s[%d:%d], s[10:11]" % (wave_lists, wave_lists + 1))
        e("  s_mov_b32 s%d, s44" % stride)
        e("  s_mov_b32 s%d, s45" % tiles)
        e("  s_mov_b64 s[%d:%d], s[46:47]" % (one_hot, one_hot + 1))
        e("  s_lshl_b32 s4, s2, 8")
        e("  s_sub_u32 s%d, s24, s4" % last)            # last row of the batch, counted from the block's first, at most 255
        e("  s_sub_u32 s%d, s%d, 1" % (last, last))
        e("  s_min_u32 s%d, s%d, 0xff" % (last, last))
        e("  s_mul_i32 s5, s4, s%d" % stride)
        e("  s_mul_hi_u32 s6, s4, s%d" % stride)
        e("  s_add_u32 s%d, s40, s5" % rows_base[0])
        e("  s_addc_u32 s%d, s41, s6" % (rows_base[0] + 1))
        e("  s_lshl_b32 s4, s%d, 6" % stride)           # 64 rows
        for j in range(1, 4):
            e("  s_add_u32 s%d, s%d, s4" % (rows_base[j], rows_base[j - 1]))
            e("  s_addc_u32 s%d, s%d, 0" % (rows_base[j] + 1, rows_base[j - 1] + 1))
        lane_piece(probe, probe + 1)
        for j in range(4):
            e("  v_add_u32_e32 v%d, %d, v%d" % (place + j, 64 * j, probe + 1))
            e("  v_cmp_ge_u32_e64 s[%d:%d], s%d, v%d" % (rows_there[j], rows_there[j] + 1, last, place + j))
        # The workgroups start with different tiles: those that run side by side would otherwise all read the same columns of
        # their rows, and rows of about 4 KB put these on few memory channels (262 000 documents, 500 trees: 431 -> 400 us).
        e("  s_mov_b32 s%d, s%d" % (left, tiles))
        e("  s_and_b32 s4, s2, 15")
        e("  s_mul_i32 s4, s4, s%d" % tiles)
        e("  s_lshr_b32 s%d, s4, 4" % following)
        e("  s_lshl_b32 s%d, s%d, 2" % (register, following))
        e("  s_lshl_b32 s4, s%d, 6" % following)
        e("  s_add_u32 s4, s4, %d" % OFFSETS_AT)
        e("  s_add_u32 s6, s%d, s4" % table)
        e("  s_addc_u32 s7, s%d, 0" % (table + 1))
        e("  v_lshlrev_b32_e32 v%d, 2, v%d" % (place, probe))
        e("  global_load_dword v%d, v%d, s[6:7]" % (offset, place))
        e("  v_mul_u32_u24_e32 v%d, 0x%x, v%d" % (tables, PIECE_BYTES, probe))
        e("  v_add_u32_e32 v%d, 0x%x, v%d" % (tables, IMAGES_AT, tables))
        e("  v_mov_b32_e32 v%d, 0x4b000000" % two_to_23)
        e("  v_sub_u32_e32 v%d, v%d, v%d" % (table_of_float, tables, two_to_23))
        copy_image(0)
        load_infos(0)
        next_tile()
        e("  s_mov_b32 s%d, 2" % two)
        e("  s_mov_b32 s%d, 0x%x" % (highest_cell, struct.unpack("<I", struct.pack("<f", grid_cells(six) - 1))[0]))
        for i in range(4):
            e("  s_mov_b32 s%d, 0" % (lists[1] + i))     # of the tile before the first
        e("  s_waitcnt vmcnt(%d)" % copies)
        load_values(0)
        e("  s_waitcnt vmcnt(4) lgkmcnt(0)")
        e("  s_barrier")
        e("%s_tiles:" % name)
        for x in range(2):
            label = "%s_tile%d" % (name, x)
            read_bins(1 - x)
            e("  v_bfe_u32 v%d, v1, 2, 4" % probe)
            e("  v_mul_u32_u24_e32 v%d, 48, v%d" % (probe, probe))
            e("  v_add_u32_e32 v%d, 0x%x, v%d" % (probe, IMAGES_AT + (x + 1) * image - PARAMETERS_BYTES, probe))
            for q in range(3):
                e("  ds_read_b128 v[%d:%d], v%d%s" % (scale + 4 * q, scale + 4 * q + 3, probe, " offset:%d" % (16 * q) if q else ""))
            copy_image(1 - x)
            e("  s_waitcnt lgkmcnt(0)")
            take_bins()
            load_values(1 - x)
            load_infos(1 - x)
            next_tile()
            e("  s_waitcnt vmcnt(%d)" % (copies + 4))  # this tile's values
            for j in (0, 2):
                search(label, x, j)
            lane_piece(place, place + 1)
            e("  v_mul_u32_u24_e32 v%d, 0x040404, v%d" % (place + 2, place))
            e("  v_lshlrev_b32_e32 v%d, 26, v%d" % (place + 3, place))
            e("  v_or_b32_e32 v%d, v%d, v%d" % (place + 2, place + 2, place + 3))
            e("  v_lshlrev_b32_e32 v%d, 2, v%d" % (place + 1, place + 1))
            e("  v_mul_u32_u24_e32 v%d, 0x%x, v%d" % (place, 4 * COLUMN_BYTES, place))
            e("  v_add_u32_e32 v%d, v%d, v%d" % (place, place, place + 1))
            for c in range(4):
                e("  v_sub_u32_e32 v%d, v%d, v%d" % (out + c, out + c, place + 2))
                e("  ds_write_b32 v%d, v%d offset:%d" % (place, out + c, BUFFERS[x] + c * COLUMN_BYTES))
            e("  s_cmp_lg_u32 s%d, 0" % (infos[x] + 1))
            e("  s_cbranch_scc1 %s_hot" % label)
            e("%s_hot_back:" % label)
            out_of_line.append(lambda label=label, x=x: one_hot_columns(label, x))
            e("  s_waitcnt vmcnt(4) lgkmcnt(0)")      # the next tile's image, the bins
            e("  s_barrier")
            for base in (tables, table_of_float):
                e("  v_%s_u32_e32 v%d, 0x%x, v%d" % ("add" if x == 0 else "subrev", base, image, base))
            e("  s_sub_u32 s%d, s%d, 1" % (left, left))
            e("  s_cmp_eq_u32 s%d, 0" % left)
            e("  s_cbranch_scc1 %s_last%d" % (name, x))
        e("  s_branch %s_tiles" % name)
        for x in range(2):
            e("%s_last%d:" % (name, x))
            read_bins(x)
            if x == 0:
                e("  s_branch %s_binarized" % name)
        e("%s_binarized:" % name)
        e("  s_waitcnt vmcnt(0) lgkmcnt(0)")
        take_bins()
        e("  v_lshrrev_b32_e32 v0, 2, v1")
        e("  s_lshl_b32 s4, s3, 6")
        e("  v_add_u32_e32 v0, s4, v0")
        e("  v_lshlrev_b32_e32 v2, 2, v1")
        # the leaf regions and slots take the images' and buffers' place
        e("  s_barrier")

    e(".text")
    e(".globl %s" % name)
    e(".p2align 8")
    e(".type %s,@function" % name)
    e("%s:" % name)
    e("  s_load_dwordx8 s[8:15], s[0:1], 0x0")      # bins, wave table, records, extra rows
    e("  s_load_dwordx8 s[16:23], s[0:1], 0x20")    # leaves, out, bias, scale
    e("  s_load_dwordx4 s[24:27], s[0:1], 0x40")    # documents, rounds, bytes of a block's bins
    e("  v_lshrrev_b32_e32 v4, 6, v0")
    e("  v_and_b32_e32 v1, 63, v0")
    e("  v_readfirstlane_b32 s3, v4")
    e("  v_lshlrev_b32_e32 v2, 4, v1")
    e("  v_lshlrev_b32_e32 v1, 2, v1")
    e("  s_mov_b32 s%d, 0x80808080" % high_bits)
    e("  s_mov_b32 s%d, 0xc0c0c0c0" % pair_bits)
    e("  s_waitcnt lgkmcnt(0)")
    if not fused:
        e("  s_mul_i32 s4, s2, s26")
        e("  s_mul_hi_u32 s5, s2, s26")
        e("  s_add_u32 s8, s8, s4")
        e("  s_addc_u32 s9, s9, s5")
    e("  s_mov_b64 s[6:7], s[12:13]")               # records to s[14:15], extra rows to s[12:13]
    e("  s_mov_b64 s[12:13], s[14:15]")
    e("  s_mov_b64 s[14:15], s[6:7]")
    for pointer, per_wave in ((10, WAVE_TABLE_BYTES), (14, RECORD_BYTES), (16, ROUND_STEPS * leaf_bytes)):
        e("  s_mul_i32 s4, s3, 0x%x" % per_wave)
        e("  s_add_u32 s%d, s%d, s4" % (pointer, pointer))
        e("  s_addc_u32 s%d, s%d, 0" % (pointer + 1, pointer + 1))
    if fused:
        binarize_tiles()
    if folded:
        e("  v_mov_b32_e32 v39, 0x%x" % (0x01010101 * (0x80 - (1 << first_bit))))
    for j in range(4):
        e("  v_mov_b32_e32 v%d, 0x%x" % (sc0 + j, (1 << (3 - first_bit)) << (8 * j)))
    for r in list(range(lv0, lv0 + 8)) + list(range(ac0, ac0 + 8)):
        e("  v_mov_b32_e32 v%d, 0" % r)
    e("  s_load_dwordx2 s[6:7], s[10:11], 0x%x" % (4 * WAVE_BUCKETS))
    e("  s_mul_i32 s4, s3, 0x%x" % (REGIONS * leaf_bytes))
    for i in range(REGIONS):
        e("  s_add_u32 s%d, s4, 0x%x" % (regions[i], SLOTS * 256 + i * leaf_bytes))
    fetch_leaves(regions[0], False)
    fetch_leaves(regions[1], True)
    if fused:
        e("  s_waitcnt lgkmcnt(0)")
    else:
        # the block's bins: the offsets of the wave's buckets take all scalar registers from 32 on for a moment
        for part in range(WAVE_BUCKETS // 16):
            e("  s_load_dwordx16 s[%d:%d], s[10:11], 0x%x" % (32 + 16 * part, 47 + 16 * part, part * 64))
        e("  s_waitcnt lgkmcnt(0)")
        for i in range(WAVE_BUCKETS):
            e("  s_add_u32 s4, s8, s%d" % (32 + i))
            e("  s_addc_u32 s5, s9, 0")
            e("  global_load_dword v%d, v1, s[4:5]" % (b0 + i))
    e("  s_add_u32 s12, s12, s6")
    e("  s_addc_u32 s13, s13, 0")
    # the groups that the first round looks at, EARLY_ROWS at a time, the first of them on their way while the bins come
    early = [32 + 16 * i for i in range(EARLY_ROWS)]

    def load_early():
        for i, regs in enumerate(early):
            e("  s_load_dwordx16 s[%d:%d], s[12:13], 0x%x" % (regs, regs + 15, i * GROUP_BYTES))
    load_early()
    load_tree_row(0)
    for p in range(8):
        e("  s_mov_b32 s%d, 0x%x" % (masks[p], 0x01010101 << p))
    e("  s_waitcnt vmcnt(0) lgkmcnt(0)")
    e("%s_first:" % name)
    for i, regs in enumerate(early):
        e("  s_cmp_eq_u32 s7, 0")
        e("  s_cbranch_scc1 %s_ready" % name)
        compare_group(regs, "%s_early%d" % (name, i))
        e("  s_sub_u32 s7, s7, 1")
        advance(12, GROUP_BYTES)
    load_early()
    e("  s_waitcnt lgkmcnt(0)")
    e("  s_branch %s_first" % name)
    e("%s_ready:" % name)
    e("  s_waitcnt lgkmcnt(0)")
    e("  s_barrier")
    read_dwords(0, [])
    load_tree_row(1)
    load_group_row(0)
    e("%s_loop:" % name)
    turn = ROUND_STEPS * REGIONS               # whole rounds after which the regions come round
    for number in range(turn):
        step(number)
        if number % ROUND_STEPS == ROUND_STEPS - 1:
            advance(14, round_record_bytes)
            e("  s_sub_u32 s25, s25, 1")
            e("  s_cmp_eq_u32 s25, 0")
            e("  s_cbranch_scc1 %s_done" % name)
    e("  s_branch %s_loop" % name)
    e("%s_done:" % name)
    e("  s_waitcnt vmcnt(0) lgkmcnt(0)")
    for line in sums():
        e(line)
    # the sixteen sums of a document, [wave][document], where the slots were: behind the last round's barrier no wave has a
    # slot to read any more (but for the reads ahead, whose dwords nobody uses)
    e("  v_lshlrev_b32_e32 v3, 1, v1")
    e("  s_lshl_b32 s4, s3, 11")
    e("  v_add_u32_e32 v3, s4, v3")
    for j in range(4):
        e("  ds_write_b64 v3, v[%d:%d] offset:%d" % (ac0 + 2 * j, ac0 + 2 * j + 1, 512 * j))
    e("  s_waitcnt lgkmcnt(0)")
    e("  s_barrier")
    e("  s_cmp_gt_u32 s3, 3")
    e("  s_cbranch_scc1 %s_end" % name)
    e("  s_load_dwordx2 s[6:7], s[20:21], 0x0")
    e("  v_lshlrev_b32_e32 v3, 3, v0")
    for w in range(WAVES):
        e("  ds_read_b64 v[%d:%d], v3 offset:%d" % (b0 + 2 * w, b0 + 2 * w + 1, 2048 * w))
    e("  s_waitcnt lgkmcnt(0)")
    for w in range(1, WAVES):
        e("  v_add_f64 v[%d:%d], v[%d:%d], v[%d:%d]" % (b0, b0 + 1, b0, b0 + 1, b0 + 2 * w, b0 + 2 * w + 1))
    e("  v_mul_f64 v[%d:%d], s[22:23], v[%d:%d]" % (b0, b0 + 1, b0, b0 + 1))
    e("  v_add_f64 v[%d:%d], v[%d:%d], s[6:7]" % (b0, b0 + 1, b0, b0 + 1))
    e("  s_lshl_b32 s4, s2, 8")
    e("  v_add_u32_e32 v4, s4, v0")
    e("  v_cmp_gt_u32_e32 vcc, s24, v4")
    e("  s_and_saveexec_b64 s[4:5], vcc")
    e("  s_mul_i32 s4, s2, 0x800")
    e("  s_mul_hi_u32 s5, s2, 0x800")
    e("  s_add_u32 s18, s18, s4")
    e("  s_addc_u32 s19, s19, s5")
    e("  global_store_dwordx2 v3, v[%d:%d], s[18:19]" % (b0, b0 + 1))
    e("%s_end:" % name)
    e("  s_endpgm")
    while out_of_line:
        out_of_line.pop(0)()
    e(".Lend_%s:" % name)
    e(".size %s, .Lend_%s-%s" % (name, name, name))
    e("")
    e(".rodata")
    e(".p2align 6")
    e(".amdhsa_kernel %s" % name)
    e("  .amdhsa_group_segment_fixed_size %d" % lds_bytes(depth, six, fused))
    e("  .amdhsa_private_segment_fixed_size 0")
    e("  .amdhsa_kernarg_size %d" % (112 if fused else 80))
    e("  .amdhsa_user_sgpr_count 2")
    e("  .amdhsa_user_sgpr_kernarg_segment_ptr 1")
    e("  .amdhsa_system_sgpr_workgroup_id_x 1")
    e("  .amdhsa_system_sgpr_workgroup_id_y 0")
    e("  .amdhsa_system_sgpr_workgroup_id_z 0")
    e("  .amdhsa_system_vgpr_workitem_id 0")
    e("  .amdhsa_next_free_vgpr %d" % vgprs)
    e("  .amdhsa_next_free_sgpr 102")
    e("  .amdhsa_accum_offset %d" % vgprs)
    e("  .amdhsa_reserve_vcc 1")
    e("  .amdhsa_float_round_mode_32 0")
    e("  .amdhsa_float_round_mode_16_64 0")
    e("  .amdhsa_float_denorm_mode_32 3")
    e("  .amdhsa_float_denorm_mode_16_64 3")
    e("  .amdhsa_dx10_clamp 1")
    e("  .amdhsa_ieee_mode 1")
    e(".end_amdhsa_kernel")
    e("")
    arguments = "".join("      - {.address_space: global, .offset: %d, .size: 8, .value_kind: global_buffer}\n" % at
                        for at in range(0, 56, 8))
    arguments += "      - {.offset: 56, .size: 8, .value_kind: by_value}\n"
    arguments += "".join("      - {.offset: %d, .size: 4, .value_kind: by_value}\n" % at for at in (64, 68, 72, 76))
    if fused:
        arguments += "".join("      - {.address_space: global, .offset: %d, .size: 8, .value_kind: global_buffer}\n" % at for at in (80, 88))
        arguments += "".join("      - {.offset: %d, .size: 4, .value_kind: by_value}\n" % at for at in (96, 100))
        arguments += "      - {.address_space: global, .offset: 104, .size: 8, .value_kind: global_buffer}\n"
    meta = """  - .agpr_count: 0
    .args:
%s    .group_segment_fixed_size: %d
    .kernarg_segment_align: 8
    .kernarg_segment_size: %d
    .max_flat_workgroup_size: %d
    .name: %s
    .private_segment_fixed_size: 0
    .sgpr_count: 108
    .sgpr_spill_count: 0
    .symbol: %s.kd
    .uniform_work_group_size: 1
    .uses_dynamic_stack: false
    .vgpr_count: %d
    .vgpr_spill_count: 0
    .wavefront_size: 64
""" % (arguments, lds_bytes(depth, six, fused), 112 if fused else 80, WAVES * 64, name, name, vgprs)
    return "\n".join(o), meta
