"""Scalar-register hazards around the asm blocks of the kernels (no GPU needed: hipcc cross-compiles).

A memory instruction or an MFMA inside an asm block is invisible to the compiler's hazard pass, so
the assembly of every kernel source is checked for (1) a vector-memory instruction reading a scalar
register that a vector-ALU instruction wrote fewer than 5 slots earlier, (2) a global->LDS copy
reading M0 right after the scalar instruction that wrote it, (3) an MFMA result touched fewer than 11
slots after the MFMA, (4) an MFMA operand written by the vector ALU fewer than 2 slots before,
(5) a dot-product result read by another vector-ALU opcode fewer than 3 slots later (or overwritten
by one fewer than 4 slots later) and (6) the destination of an asm block's global load touched before a
wait that covers the load.
The checker itself is pinned on hand-written listings."""
import isa_lint

HAZ_VMEM = """
	v_readfirstlane_b32 s17, v210
	v_readfirstlane_b32 s16, v211
	;;#ASMSTART
	global_load_dwordx4 v[152:155], v212, s[16:17]
	;;#ASMEND
"""
OK_NOPS = HAZ_VMEM.replace(";;#ASMSTART", "s_nop 4\n\t;;#ASMSTART")
SHORT_NOPS = HAZ_VMEM.replace(";;#ASMSTART", "s_nop 2\n\t;;#ASMSTART")
OK_SALU = HAZ_VMEM.replace(";;#ASMSTART", "s_mov_b64 s[16:17], s[16:17]\n\t;;#ASMSTART")
OK_OTHER_REG = HAZ_VMEM.replace("s[16:17]", "s[18:19]")
HAZ_CMP = """
	v_cmp_lt_u32_e64 s[4:5], v1, v2
	v_mov_b32_e32 v3, 0
	buffer_load_dword v4, v5, s[4:7], 0 offen
"""
HAZ_M0 = """
	s_add_i32 m0, s38, 0x2000
	global_load_lds_dwordx4 v191, s[26:27]
"""
OK_M0 = HAZ_M0.replace("\tglobal_load_lds", "\ts_nop 0\n\tglobal_load_lds")
OK_M0_PLAIN_LOAD = HAZ_M0.replace("global_load_lds_dwordx4 v191", "global_load_dwordx4 v[0:3], v191")


MFMA = "\tv_mfma_f32_32x32x16_f16 v[32:47], v[6:9], v[116:119], v[32:47]\n"
MFMA_READ_EARLY = MFMA + "\tv_add_f32_e32 v1, v2, v3\n" * 9 + "\tv_exp_f32_e32 v0, v33\n"
MFMA_READ_OK = MFMA + "\tv_add_f32_e32 v1, v2, v3\n" * 11 + "\tv_exp_f32_e32 v0, v33\n"
MFMA_READ_NOPS = MFMA + "\ts_nop 7\n\ts_nop 2\n\tv_exp_f32_e32 v0, v33\n"
MFMA_CHAIN_OK = MFMA + "\tv_mfma_f32_32x32x16_f16 v[32:47], v[10:13], v[120:123], v[32:47]\n"
MFMA_AS_OPERAND = MFMA + "\tv_mfma_f32_32x32x16_f16 v[48:63], v[32:35], v[120:123], v[48:63]\n"
VALU_THEN_MFMA = "\tv_cvt_pkrtz_f16_f32 v6, v1, v2\n" + MFMA
VALU_THEN_MFMA_OK = "\tv_cvt_pkrtz_f16_f32 v6, v1, v2\n\ts_nop 1\n" + MFMA


def test_checker_on_matrix_core_listings():
    assert len(isa_lint.lint(MFMA_READ_EARLY)) == 1
    assert isa_lint.lint(MFMA_READ_OK) == []
    assert isa_lint.lint(MFMA_READ_NOPS) == []
    assert isa_lint.lint(MFMA_CHAIN_OK) == []
    assert len(isa_lint.lint(MFMA_AS_OPERAND)) == 1
    assert len(isa_lint.lint(VALU_THEN_MFMA)) == 1
    assert isa_lint.lint(VALU_THEN_MFMA_OK) == []


def test_checker_on_transcendental_results():
    assert len(isa_lint.lint("\tv_exp_f32_e32 v1, v2\n\tv_mul_f32_e32 v3, v1, v4\n")) == 1
    assert isa_lint.lint("\tv_exp_f32_e32 v1, v2\n\tv_exp_f32_e32 v3, v1\n") == []
    assert isa_lint.lint("\tv_exp_f32_e32 v1, v2\n\tv_mul_f32_e32 v1, v5, v4\n") == []
    assert isa_lint.lint("\tv_exp_f32_e32 v1, v2\n\ts_nop 0\n\tv_mul_f32_e32 v3, v1, v4\n") == []


def test_checker_on_dot_product_results():
    dot = "\tv_dot2_f32_f16 v80, v24, s36, 0\n"
    acc = "\tv_dot2_f32_f16 v80, v25, s36, v80\n"
    # the same opcode accumulating into its own result is forwarded
    assert isa_lint.lint(dot + acc) == []
    # another opcode reading the sum: three idle slots needed
    assert len(isa_lint.lint(dot + acc + "\tv_cmp_nge_f32_e32 vcc, s37, v80\n")) == 1
    assert len(isa_lint.lint(dot + acc + "\ts_nop 1\n\tv_cmp_nge_f32_e32 vcc, s37, v80\n")) == 1
    assert isa_lint.lint(dot + acc + "\ts_nop 2\n\tv_cmp_nge_f32_e32 vcc, s37, v80\n") == []
    # the two-operand form accumulating into the result of the three-operand form is another opcode
    assert len(isa_lint.lint(dot + "\tv_dot2c_f32_f16_e32 v80, s36, v25\n")) == 1
    assert isa_lint.lint("\tv_dot2c_f32_f16_e32 v80, s36, v24\n\tv_dot2c_f32_f16_e32 v80, s36, v25\n") == []
    # the same opcode taking the sum as a multiplicand
    assert len(isa_lint.lint(dot + "\tv_dot2_f32_f16 v81, v80, s36, 0\n")) == 1
    # overwritten by another opcode within four slots
    assert len(isa_lint.lint(dot + "\tv_add_f32_e32 v1, v2, v3\n" * 3 + "\tv_mov_b32_e32 v80, 0\n")) == 1
    assert isa_lint.lint(dot + "\tv_add_f32_e32 v1, v2, v3\n" * 4 + "\tv_mov_b32_e32 v80, 0\n") == []


def test_checker_on_hand_written_listings():
    assert len(isa_lint.lint(HAZ_VMEM)) == 1
    assert len(isa_lint.lint(SHORT_NOPS)) == 1
    assert isa_lint.lint(OK_NOPS) == []
    assert isa_lint.lint(OK_SALU) == []
    assert isa_lint.lint(OK_OTHER_REG) == []
    assert len(isa_lint.lint(HAZ_CMP)) == 1
    assert len(isa_lint.lint(HAZ_M0)) == 1
    assert isa_lint.lint(OK_M0) == []
    assert isa_lint.lint(OK_M0_PLAIN_LOAD) == []


def test_kernel_sources_have_no_scalar_register_hazards():
    report = isa_lint.analyse_sources()
    assert set(report) == set(isa_lint._build.SOURCES)
    assert {s: h for s, (h, _) in report.items() if h} == {}
    # the hand-scheduled kernels keep everything in registers: a reload would make the compiler wait for
    # every memory operation in flight, the stage copies included, in the middle of the schedule
    for src in ("fta_fwd1.hip", "fta_fwd1_slabs.hip", "fta_fwd2.hip", "fta_bwd_dq1.hip", "fta_bwd_dq1_bf16.hip", "fta_bwd_dkdv1.hip",
                "fta_bwd_dkdv1_bf16.hip", "fta_bwd_short.hip"):
        spilling = dict(report[src][1])
        if src == "fta_fwd2.hip":
            # known: the tail-masking instances of the two-slab D=64 forward (template arguments <T, 2, true>)
            # keep five bias registers of a row's last tile in scratch (three reloads per row)
            spilling = {k: v for k, v in spilling.items() if "Li2ELb1E" not in k}
        if src == "fta_bwd_short.hip":
            # known: its widest instances with dropout (eight waves, D=32) keep a few values of a row in scratch; every reload
            # waits for the next row's copies, which are in flight from the row's start
            assert all(v <= 17 for k, v in spilling.items() if "Li32ELi8ELb1E" in k)
            spilling = {k: v for k, v in spilling.items() if "Li32ELi8ELb1E" not in k}
        if src.startswith("fta_bwd_dkdv1"):
            # known: the D=64 instances for 384 queries per launch (template arguments <T, 64, 12, 4, ...>) use
            # every vector and accumulation register and keep one loop-invariant pair in scratch (one
            # reload per row; three accesses per kernel); still 2.5x the general kernel's rate at that length
            assert all(v <= 3 for k, v in spilling.items() if "Li64ELi12ELi4E" in k)
            spilling = {k: v for k, v in spilling.items() if "Li64ELi12ELi4E" not in k}
        assert spilling == {}, f"{src}: kernels that spill registers"
    # the general forward without dropout, whose copies are in flight in the same way
    for src in ("fta_fwd.hip", "fta_fwd_feat.hip"):
        spilling = {k: v for k, v in report[src][1].items() if "fta_fwd_kernel" in k and "ELb0ELi" in k}
        # known: the D=64 instance of 448-key slabs stores five values and reads them back twice per row
        assert all(v <= 10 for k, v in spilling.items() if "Li64ELi14E" in k)
        assert {k: v for k, v in spilling.items() if "Li64ELi14E" not in k} == {}, f"{src}: kernels that spill registers"
    # with dropout: slabs of 384 and 448 keys at D=32 spill and are the faster for it; 512 keys, and 256 at D=64, may keep values of a
    # row there, but no offsets of the copies that every stage would reload (104 and 30 accesses with them)
    spilling = {k: v for k, v in report["fta_fwd_feat.hip"][1].items() if "fta_fwd_kernel" in k and "ELb1ELi" in k}
    assert all(v <= 30 for k, v in spilling.items() if "Li32ELi16E" in k)
    assert all(v <= 8 for k, v in spilling.items() if "Li64E" in k.split("ELb1E")[1][:5])


def test_checker_counts_the_scratch_accesses_of_a_kernel():
    listing = ("_Zspills:\n\tscratch_store_dword off, v51, off offset:4\n\tv_mov_b32 v1, v2\n\tscratch_load_dword v88, off, off offset:4\n"
               "\t.end_amdhsa_kernel\n_Zclean:\n\tv_mov_b32 v1, v2\n\t.end_amdhsa_kernel\n")
    assert isa_lint.scratch_ops(listing) == {"_Zspills": 2}


def test_checker_on_wide_store_data():
    bad = "global_store_dwordx4 v131, v[34:37], s[10:11]\nv_mul_f32_e32 v34, v8, v38\n"
    late = "global_store_dwordx4 v131, v[34:37], s[10:11]\ns_nop 1\nv_mul_f32_e32 v34, v8, v38\n"
    other = "global_store_dwordx4 v131, v[34:37], s[10:11]\nv_mul_f32_e32 v40, v8, v38\nv_mul_f32_e32 v131, v8, v38\n"
    narrow = "global_store_dwordx2 v131, v[34:35], s[10:11]\nv_mul_f32_e32 v34, v8, v38\n"
    assert len(isa_lint.lint(bad)) == 1
    assert isa_lint.lint(late) == [] and isa_lint.lint(other) == [] and isa_lint.lint(narrow) == []


def _asm(line):
    return f"\t;;#ASMSTART\n\t{line}\n\t;;#ASMEND\n"


def test_checker_on_loads_that_the_compiler_does_not_see():
    load = _asm("global_load_dwordx4 v[8:11], v1, s[2:3] offset:16")
    copy = _asm("global_load_lds_dwordx4 v2, s[4:5]")
    add, wait = "\tv_pk_add_f16 v12, v9, v13\n", "\ts_waitcnt vmcnt({})\n"
    assert len(isa_lint.lint(load + add)) == 1
    assert isa_lint.lint(load + wait.format(0) + add) == []
    # the loads of ordinary code have the compiler's own waits
    assert isa_lint.lint("\tglobal_load_dwordx4 v[8:11], v1, s[2:3]\n\ts_waitcnt lgkmcnt(0)\n" + add) == []
    # a wait that lets more operations stay in flight than were issued behind the load
    assert len(isa_lint.lint(load + copy * 2 + wait.format(3) + add)) == 1
    assert isa_lint.lint(load + copy * 3 + wait.format(3) + add) == []
    # moved, spilled or overwritten before it is there
    assert len(isa_lint.lint(load + "\tv_accvgpr_write_b32 a0, v10\n")) == 1
    assert len(isa_lint.lint(load + "\tscratch_store_dword off, v11, off\n")) == 1
    assert len(isa_lint.lint(load + "\tv_mov_b32_e32 v8, 0\n")) == 1
    assert len(isa_lint.lint(_asm("global_load_dwordx4 a[8:11], v1, s[2:3]") + "\tv_accvgpr_read_b32 v0, a8\n")) == 1
    # over the back edge of a loop: the reader stands in front of the load
    loop = "\ts_nop 0\n.LBB0_1:\n{}" + add + load + "\ts_cbranch_scc1 .LBB0_1\n" + wait.format(0) + "\ts_endpgm\n"
    assert len(isa_lint.lint(loop.format(""))) == 1
    assert isa_lint.lint(loop.format(wait.format(0))) == []
    # one of two ways round the wait
    assert len(isa_lint.lint(load + "\ts_cbranch_execz .LBB0_2\n" + wait.format(0) + ".LBB0_2:\n" + add)) == 1
    assert isa_lint.lint(load + "\ts_branch .LBB0_2\n" + add + ".LBB0_2:\n" + wait.format(0) + add) == []


def test_checker_on_records_between_waves():
    kernel = "_ZN3fta19fta_bwd_dq1w_kernelX:\n{}\ts_endpgm\n\t.end_amdhsa_kernel\n"
    read, write, barrier = "\tds_read_b128 v[0:3], v9 offset:0x800\n", "\tds_write_b128 v8, a[0:3]\n", "\ts_barrier\n"
    operand = "\tds_read_b128 v[4:7], v9 offset:0x4000\n"
    assert isa_lint.exchange_kernels(kernel.format("")) == ["_ZN3fta19fta_bwd_dq1w_kernelX"]
    assert len(isa_lint.lint(kernel.format(read + operand + write))) == 1
    assert isa_lint.lint(kernel.format(read + barrier + write)) == []
    assert isa_lint.lint(kernel.format(barrier + write + operand + barrier + read)) == []
    # the next row's write, over the back edge of the row loop, and the last row's, behind the loop
    loop = ".LBB0_1:\n{}" + write + barrier + read + "{}\ts_cbranch_scc1 .LBB0_1\n{}" + write + barrier + read
    assert isa_lint.lint(kernel.format(loop.format("", barrier, ""))) == []
    assert isa_lint.lint(kernel.format(loop.format(barrier, "", barrier))) == []
    assert len(isa_lint.lint(kernel.format(loop.format("", "", barrier)))) == 1
    assert len(isa_lint.lint(kernel.format(loop.format(barrier, "", "")))) == 1
    # a kernel that is named but has no exchange in a form that the checker knows
    assert len(isa_lint.lint(kernel.format(operand + barrier))) == 1
    # the kernel for head dim 32, whose records are moved by pairs of floats; with one slab it has none
    floats = kernel.replace("_ZN3fta19fta_bwd_dq1w_kernelX", "_ZN3fta18fta_bwd_dq1_kernelINS_3F16ELi32ELi2ELi5E")
    read, write = "\tds_read2st64_b32 v[0:1], v9 offset1:1\n", "\tds_write2st64_b32 v8, v2, v3 offset1:1\n"
    assert len(isa_lint.lint(floats.format(read + write))) == 1
    assert isa_lint.lint(floats.format(write + barrier + read + barrier + write)) == []
    assert isa_lint.lint(floats.replace("Li32ELi2E", "Li32ELi1E").format("")) == []
    # other kernels hand nothing over in this way
    assert isa_lint.lint(kernel.replace("dq1w", "dkdv").format(read + write)) == []
