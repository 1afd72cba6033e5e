"""Register and scratch budget of the tuned kernels, read from the metadata of the device code inside the built
library (no GPU needed): a kernel that starts to spill into scratch memory inside its tile loop loses tens of
percent without failing any parity test, so the budget is pinned here.  The code objects are taken out of the
library's .hip_fatbin section with the ROCm LLVM tools (one offload bundle per translation unit)."""
import os
import re
import shutil
import subprocess

import pytest

from dmf_amd import _lib

LLVM = "/opt/rocm/llvm/bin"
TOOLS = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf", "llvm-objdump")]
pytestmark = pytest.mark.skipif(not all(os.path.exists(t) for t in TOOLS), reason="ROCm LLVM tools not installed")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    """Paths of the device code objects of the built library."""
    lib = _lib.LIB_PATH
    if not os.path.exists(lib):
        pytest.skip("library not built")
    tmp = tmp_path_factory.mktemp("codeobj")
    fat = tmp / "fat.bin"
    subprocess.run([TOOLS[0], f"--dump-section=.hip_fatbin={fat}", lib, str(tmp / "discard.so")], check=True)
    data = fat.read_bytes()
    starts = [m.start() for m in re.finditer(re.escape(MAGIC), data)]
    assert starts, "no offload bundle in the library"
    objects = []
    for i, s in enumerate(starts):
        bundle, co = tmp / f"b{i}.bin", tmp / f"co{i}.elf"
        bundle.write_bytes(data[s:starts[i + 1] if i + 1 < len(starts) else len(data)])
        subprocess.run([TOOLS[1], "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={bundle}", f"--output={co}",
                        "--unbundle"], check=True)
        objects.append(str(co))
    yield objects
    shutil.rmtree(tmp, ignore_errors=True)


@pytest.fixture(scope="module")
def kernels(code_objects):
    """{mangled kernel name: {vgpr_count, vgpr_spill_count, private_segment_fixed_size, group_segment_fixed_size}}"""
    out = {}
    for co in code_objects:
        notes = subprocess.run([TOOLS[2], "--notes", co], check=True, capture_output=True, text=True).stdout
        for m in re.finditer(r"\.name:\s+(\S+)\n(.*?)\.wavefront_size", notes, re.S):
            fields = dict(re.findall(r"\.(\w+):\s+(\d+)", m.group(2)))
            out[m.group(1)] = {k: int(v) for k, v in fields.items()}
    return out


def _fwd(D, jvp, nw, qn=False, kn=False):
    b = lambda x: "1" if x else "0"
    return f"_ZN3dmf20attn_fwd_bf16_kernelILi{D}ELb{b(jvp)}ELi{nw}ELb{b(qn)}ELb{b(kn)}EEEvNS_9FwdParamsE"


def test_every_tuned_kernel_is_in_the_library(kernels):
    for D in (64, 72, 80, 96, 128):
        for jvp in (False, True):
            assert _fwd(D, jvp, 8) in kernels and _fwd(D, jvp, 4) in kernels
        assert f"_ZN3dmf23attn_bwd_dq_bf16_kernelILi{D}ELi2EEEvNS_9BwdParamsE" in kernels
        assert f"_ZN3dmf24attn_bwd_dkv_bf16_kernelILi{D}ELi4EEEvNS_9BwdParamsE" in kernels
    for D in (64, 72, 80, 96):
        assert f"_ZN3dmf26attn_bwd_fused_bf16_kernelILi{D}EEEvNS_9BwdParamsE" in kernels


@pytest.mark.parametrize("D", [64, 72, 80])
def test_model_head_dims_do_not_spill(kernels, D):
    """Head dims 64 and 72 are the model's (DMFT-B/2, -XL/2), 80 shares their code shape: no vector register of any
    tuned forward or backward kernel goes to scratch memory, with or without the in-kernel q / k norm."""
    names = [n for n in kernels if re.search(rf"attn_(fwd|bwd_dq|bwd_dkv|bwd_fused)_bf16_kernelILi{D}E", n)]
    assert len(names) >= 8
    for n in names:
        assert kernels[n]["vgpr_spill_count"] == 0, (n, kernels[n])


def test_benchmark_kernels_fit_two_waves_per_simd_without_scratch(kernels):
    """The six kernels the bench line reports (head dim 72): at most 256 VGPRs (two waves per SIMD for the 8-wave
    work-groups), no spills, no private segment."""
    names = [_fwd(72, True, 8), _fwd(72, False, 8), "_ZN3dmf23attn_bwd_dq_bf16_kernelILi72ELi2EEEvNS_9BwdParamsE",
             "_ZN3dmf24attn_bwd_dkv_bf16_kernelILi72ELi4EEEvNS_9BwdParamsE", "_ZN3dmf26attn_bwd_fused_bf16_kernelILi72EEEvNS_9BwdParamsE"]
    for n in names:
        k = kernels[n]
        assert k["vgpr_count"] <= 256 and k["vgpr_spill_count"] == 0 and k["private_segment_fixed_size"] == 0, (n, k)
    assert kernels[_fwd(72, False, 8)]["vgpr_count"] <= 128    # primal forward: four waves per SIMD


def test_head_dim_128_forward_jvp_keeps_its_operands_out_of_scratch(kernels):
    """Head dim 128 with tangents parks its last Q / dQ operand chunks in LDS instead of spilling (8-wave work-groups)."""
    k = kernels[_fwd(128, True, 8)]
    assert k["vgpr_spill_count"] == 0 and k["private_segment_fixed_size"] == 0, k


def test_lds_budgets(kernels):
    """Static LDS is not used by the tuned kernels (their tiles are dynamic LDS, opted in per launch) and nothing
    declares more than the 160 KB of a CU."""
    for n, k in kernels.items():
        assert k.get("group_segment_fixed_size", 0) <= 160 * 1024, (n, k)


# (pattern of the mangled name, most vector registers, most spilled ones): what the launch bounds of the other kernels with a register
# plan allow -- 256 where two waves share a SIMD, 128 where four do -- and the few spills that were measured to cost less than they save
BUDGETS = [
    (r"13linear_kernelI", 256, 0), (r"18linear_walk_kernelI", 512, 0), (r"19linear_wgrad_kernelE", 256, 0), (r"17modulation_kernelI", 512, 0),
    (r"19linear_dgrad_kernelI", 512, 0), (r"24linear_wgrad_wide_kernelE", 512, 0),
    (r"23linear_walk_wide_kernelI", 512, 0), (r"22linear_walk_pre_kernelI", 512, 0),
    (r"21attn_fwd_small_kernelIDF16_Li(64|72|80|96)ELb0E", 256, 0), (r"21attn_fwd_small_kernelIDF16bLi(64|72|80|96)ELb0ELb0E", 256, 0),
    (r"21attn_fwd_small_kernelI", 512, 0),
    (r"20attn_fwd_wide_kernelIDF16_Li(72|80)ELb0E", 128, 1), (r"20attn_fwd_wide_kernelI(DF16_Li(72|80)|fLi(32|64))ELb1E", 256, 0),
    (r"18attn_bwd_dq_kernelI(f|DF16_)Li64E", 256, 0), (r"19attn_bwd_dkv_kernelIDF16_Li(64|72|80)E", 256, 0), (r"19attn_bwd_dkv_kernelIfLi64E", 256, 12),
    (r"18attn_bwd_dq_kernelI(f|DF16_)Li72E", 512, 0), (r"19attn_bwd_dkv_kernelIfLi72E", 512, 0),
]


@pytest.mark.parametrize("pattern,registers,spills", BUDGETS)
def test_products_and_split_operand_kernels_stay_within_their_launch_bounds(kernels, pattern, registers, spills):
    names = [n for n in kernels if re.search(pattern, n)]
    assert names, pattern
    for n in names:
        k = kernels[n]
        assert k["vgpr_count"] <= registers and k["vgpr_spill_count"] <= spills, (n, k)


def test_every_product_kernel_is_launched_by_a_test(kernels):
    """The kernels of dmf_linear_fwd, by their template arguments, against those that the sizes of the GPU tests reach on 256 CUs (what a
    process without a GPU plans for)."""
    from test_linear_gpu import REACHED, planned
    numbers = lambda pattern, name: tuple(int(n) for n in re.findall(pattern, name))
    built = {numbers(r"Li(\d+)E", n) for n in kernels if re.search(r"linear_(walk_)?kernelI", n)}
    reached = {numbers(r"\b(\d+)\b", planned(*size, *mode)) for _, size, modes in REACHED for mode in modes}
    assert len(built) == 16 and reached == built


# ---- LDS reads written in assembly -------------------------------------------------------------------------------------------
# The compiler takes the result of an assembly read for there at once; the hardware does not hold back an instruction that uses the register
# before the read has returned.  What keeps them apart is a wait in the source, and that the compiler moves nothing in between: checked on
# the code it made, over all paths.

SCALAR = 1 << 1024   # (a scalar load in the queue: those return in any order)


def _registers(text):
    mask = 0
    for kind, one, first, last in re.findall(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])", text):
        for r in range(int(one or first), int(one or last) + 1):
            mask |= 1 << (r + (0 if kind == "v" else 512))
    return mask


def _decode(lines, counter="lgkmcnt"):
    """(operation, registers it names, branch target, count of `counter` waited for, registers a queued read returns or None) of every
    instruction.  vmcnt: loads from memory, and those into LDS and stores, which return nothing; loads return in order, so that one may name
    the register that another is about to write as its own result."""
    code = [(int(m.group(3), 16), m.group(1), m.group(2)) for m in (re.match(r"\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):", l) for l in lines) if m]
    at, out = {a: i for i, (a, _, _) in enumerate(code)}, []
    for address, op, args in code:
        target = wait = queued = None
        names = _registers(args)
        if op == "s_branch" or op.startswith("s_cbranch"):
            offset = int(args.split()[0])
            target = at[address + 4 + 4 * (offset - 65536 * (offset >= 32768))]
        elif op == "s_waitcnt":
            assert "cnt(" in args, args
            m = re.search(counter + r"\((\d+)\)", args)
            wait = int(m.group(1)) if m else None
        elif counter == "vmcnt":
            if op.startswith(("buffer_load", "buffer_store", "global_load", "global_store", "scratch_load", "scratch_store", "global_atomic", "buffer_atomic")):
                queued = 0
                if "load" in op and not re.search(r"\blds\b", args) and "_lds_" not in op:
                    queued, names = _registers(args.split(",")[0]), _registers(args.split(",", 1)[1])
        elif op.startswith("ds_"):
            queued = _registers(args.split(",")[0]) if any(s in op for s in ("read", "_rtn", "permute", "swizzle")) else 0
        elif op.startswith(("s_load", "s_buffer_load", "s_memtime", "s_memrealtime")):
            queued = SCALAR
        assert not op.startswith(("flat_", "s_swappc", "s_setpc", "s_call")), op
        out.append((op, names, target, wait, queued))
    return out


def _touched_in_flight(code, most=16):
    """Indices of instructions that name a register a read may still be about to write.  State at a place: what the last `most` requests
    return (the counter holds no more), newest last, joined over the paths that lead there."""
    entries = {0} | {t for _, _, t, _, _ in code if t is not None} | {i + 1 for i, c in enumerate(code) if c[2] is not None}
    states, work, bad = {0: ()}, [0], set()

    def join(i, queue):
        old = states.get(i)
        if old is not None:
            n = max(len(old), len(queue))
            queue = tuple(a | b for a, b in zip((0,) * (n - len(old)) + old, (0,) * (n - len(queue)) + queue))
        if queue != old:
            states[i] = queue
            work.append(i)

    while work:
        i = work.pop()
        queue, first = states[i], True
        while first or i not in entries:
            first = False
            op, names, target, wait, queued = code[i]
            pending = 0
            for q in queue:
                pending |= q
            if names & pending:
                bad.add(i)
            if wait == 0:
                queue = ()
            elif wait is not None and not pending & SCALAR:
                queue = queue[-wait:]
            if queued is not None:
                queue = (queue + (queued,))[-most:]
            if target is not None:
                join(target, queue)
            if op in ("s_branch", "s_endpgm"):
                break
            i += 1
        else:
            join(i, queue)
    return bad


def test_the_check_sees_a_read_that_is_not_waited_for():
    lines = lambda *ops: [f"\t{op} // {4 * i:012X}: 00000000" for i, op in enumerate(ops)]
    read, use = "ds_read_b128 v[4:7], v0", "v_mov_b32_e32 v8, v5"
    assert _touched_in_flight(_decode(lines(read, use, "s_endpgm"))) == {1}
    assert not _touched_in_flight(_decode(lines(read, "s_waitcnt lgkmcnt(0)", use, "s_endpgm")))
    assert _touched_in_flight(_decode(lines(read, "ds_write_b64 v1, v[2:3]", "s_waitcnt vmcnt(0) lgkmcnt(2)", use, "s_endpgm"))) == {3}
    assert not _touched_in_flight(_decode(lines(read, "ds_write_b64 v1, v[2:3]", "s_waitcnt vmcnt(0) lgkmcnt(1)", use, "s_endpgm")))
    # over a back edge: read at the end of one turn, waited for in the next one only behind the use
    assert _touched_in_flight(_decode(lines(use, "s_waitcnt lgkmcnt(0)", read, "s_cbranch_scc1 65532", "s_endpgm"))) == {0}


def test_no_register_is_touched_between_a_product_kernels_load_and_the_wait(code_objects):
    """The bias of a walking kernel's tile is loaded in assembly and waited for by counting the requests behind it: as for the LDS reads below."""
    lines = lambda *ops: [f"\t{op} // {4 * i:012X}: 00000000" for i, op in enumerate(ops)]
    load, use, dma = "buffer_load_dword v5, v0, s[0:3], 0 offen", "v_mov_b32_e32 v8, v5", "buffer_load_dwordx4 v1, s[0:3], 0 offen lds"
    assert _touched_in_flight(_decode(lines(load, dma, "s_waitcnt vmcnt(2)", use, "s_endpgm"), "vmcnt"), 64) == {3}
    assert not _touched_in_flight(_decode(lines(load, dma, "s_waitcnt vmcnt(1)", use, "s_endpgm"), "vmcnt"), 64)
    checked = 0
    for co in code_objects:
        name, code = "", {}
        for line in subprocess.run([TOOLS[3], "-d", co], check=True, capture_output=True, text=True).stdout.splitlines():
            m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            name = m.group(1) if m else name
            code.setdefault(name, []).append(line)
        for name, lines in code.items():
            if re.search(r"linear_(walk|walk_wide|walk_pre|dgrad|wgrad_wide)_kernel", name):
                checked += 1
                assert not _touched_in_flight(_decode(lines, "vmcnt"), 64), name
    assert checked >= 17


def test_no_register_is_touched_between_its_lds_read_and_the_wait(code_objects):
    names, code = [], []
    for co in code_objects:
        for line in subprocess.run([TOOLS[3], "-d", co], check=True, capture_output=True, text=True).stdout.splitlines():
            m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if m:
                names.append(m.group(1))
                code.append([])
            elif code:
                code[-1].append(line)
    assert any("linear_walk_kernel" in n for n in names)
    for name, lines in zip(names, code):
        assert not _touched_in_flight(_decode(lines)), name
