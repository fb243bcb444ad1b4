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

What bounds it: LDS. Per tree and 256 documents 34 vector and 26 scalar instructions, and 61 LDS cycles (the dwords of eight groups
and the group's own 9 or more, four gathers 36, half of them bank conflicts, 16 for the 2 KB of leaf values) of the 75 that
a step of sixteen waves takes for each; the pair-tile kernel, in which only 128 documents share a copy of the leaf values
and every level reads its bins, 82 vector instructions and 78 LDS cycles of 115. 262 144 documents x 5000 trees x 1016
buckets 0.70 ms; with half of the leaf values' copies left out 0.60, without the gathers 0.60, without reading the groups' dwords
0.59, without the barriers 0.68, without loading rows 0.69. Tried: every request in the step that waits for it 0.77, slots
addressed by vector registers (nine more vector instructions) 0.72, leaf values through registers and ds_write_b128 0.78, one
tree in four gathered from global memory 0.70. Some 13 us per workgroup go to its start (the bins, the first groups) and end.

Kernel arguments (80 bytes):
   0 bins const uint32* [docBlock][bucketCount][64]      8 wave table const uint32* [16][80]
  16 records const uint32* [rounds + 1][16][96]         24 extra group rows const uint32*
  32 leaves const double* [rounds + 1][16][4][1 << DEPTH]   40 out double* [docCount]
  48 bias const double*                                 56 scale double
  64 docCount uint32   68 rounds uint32 (>= 1)   72 bytes of a document block's bins uint32
grid = document blocks, 1024 threads; LDS: the slots, then sixteen times three leaf regions; at the end the partial sums.
"""

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

SHAPES = [(depth, six) for depth in (8, 6) for six in (False, True)]


def kernel_name(depth, six):
    return "cbamd_eval_exchange_d%d%s" % (depth, "_s" if six else "")


def lds_bytes(depth):
    return SLOTS * 256 + WAVES * REGIONS * (8 << depth)


def gen_kernel(depth, six):
    name = kernel_name(depth, six)
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
    for j in range(4):
        e("  v_mov_b32_e32 v%d, 0x%x" % (sc0 + j, (1 << (3 - first_bit)) << (8 * j)))
    for r in list(range(lv0, lv0 + 8)) + list(range(ac0, ac0 + 8)):
        e("  v_mov_b32_e32 v%d, 0" % r)
    e("  s_mov_b32 s%d, 0x80808080" % high_bits)
    e("  s_mov_b32 s%d, 0xc0c0c0c0" % pair_bits)
    e("  s_waitcnt lgkmcnt(0)")
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
    e("  s_load_dwordx2 s[6:7], s[10:11], 0x%x" % (4 * WAVE_BUCKETS))
    e("  s_mul_i32 s4, s3, 0x%x" % (REGIONS * leaf_bytes))
    for i in range(REGIONS):
        e("  s_add_u32 s%d, s4, 0x%x" % (regions[i], SLOTS * 256 + i * leaf_bytes))
    fetch_leaves(regions[0], False)
    fetch_leaves(regions[1], True)
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
    e("  .amdhsa_group_segment_fixed_size %d" % lds_bytes(depth))
    e("  .amdhsa_private_segment_fixed_size 0")
    e("  .amdhsa_kernarg_size 80")
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
    meta = """  - .agpr_count: 0
    .args:
%s    .group_segment_fixed_size: %d
    .kernarg_segment_align: 8
    .kernarg_segment_size: 80
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
""" % (arguments, lds_bytes(depth), WAVES * 64, name, name, vgprs)
    return "\n".join(o), meta
