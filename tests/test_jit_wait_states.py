"""Wait states of four-wave bodies (csrc/quad_kernel.hpp), run-time compiled and the ahead-of-time 384-row tiles, read
from the gfx950 assembly of the code objects built here.  Their matrix instructions are inline asm, for which the compiler inserts no wait states:
a VALU write of an operand has to lie two wait states ahead of the matrix instruction that reads it, and an
accumulator may be touched 11 (16x16x128) or 19 (32x32x16) after the one that wrote it.  K of one, two and three
stages is the form in which the loop becomes straight-line code that the compiler may move instructions along."""
import ctypes
import os
import re
import subprocess

import pytest

from deep_gemm import _lib
from test_jit import _args

LLVM = '/opt/rocm/llvm/bin/'
OBJDUMP = LLVM + 'llvm-objdump'
OPERAND_WAIT, RESULT_WAIT = 2, {'16x16': 11, '32x32': 19}


def _registers(text):
    """{('v', 4), ('a', 0), ..} named by one operand."""
    m = re.match(r'([va])\[(\d+):(\d+)\]', text) or re.match(r'([va])(\d+)()\b', text)
    if m is None:
        return frozenset()
    return frozenset((m[1], i) for i in range(int(m[2]), int(m[3] or m[2]) + 1))


class _Instruction:
    def __init__(self, op, operands, address):
        self.op, self.address = op, address
        self.regs = [_registers(x) for x in operands]
        self.mfma = op.startswith('v_mfma')
        self.valu = op.startswith('v_') and not self.mfma
        # (a permlane swap writes both of its operands; compares and readfirstlane write no vector register)
        both = 'swap' in op
        self.writes = frozenset().union(*self.regs[:2 if both else 1]) if self.valu and self.regs else frozenset()
        self.touched = frozenset().union(*self.regs) if self.regs else frozenset()
        self.states = int(operands[0], 0) + 1 if op == 's_nop' else 1


def _parse(listing):
    """Instructions of one function and, for each, the indices that run right before it."""
    code, target = [], {}
    for line in listing.splitlines():
        m = re.match(r'\s+(\S+)\s*(.*?)\s*// ([0-9A-F]{12}):', line)
        if m is None:
            continue
        operands = [x.strip() for x in re.split(r',\s*(?![^\[]*\])', m[2])] if m[2] else []
        if operands and operands[0].split()[0:1]:
            operands = [x.split()[0] if x else x for x in operands]
        code.append(_Instruction(m[1], operands, int(m[3], 16)))
        t = re.search(r'<[^>]*\+0x([0-9a-f]+)>$', line.strip())
        if m[1].startswith(('s_branch', 's_cbranch')):
            assert t is not None, line
            target[len(code) - 1] = int(t[1], 16)
    start = code[0].address
    at = {x.address - start: i for i, x in enumerate(code)}
    before = [[i - 1] if i and code[i - 1].op not in ('s_branch', 's_endpgm') else [] for i in range(len(code))]
    for i, offset in target.items():
        before[at[offset]].append(i)
    return code, before


def _writers_within(code, before, i, states, hit):
    """Instructions fewer than `states` wait states ahead of instruction i for which hit() holds."""
    found, todo, seen = [], [(p, 0) for p in before[i]], {}
    while todo:
        p, gap = todo.pop()
        if gap >= states or seen.get(p, states) <= gap:
            continue
        seen[p] = gap
        if hit(code[p]):
            found.append((code[p], gap))
        todo += [(x, gap + code[p].states) for x in before[p]]
    return found


def violations(listing):
    code, before = _parse(listing)
    out, count = [], 0
    # (most instructions have neither a matrix instruction nor a branch target close behind them: nothing to follow)
    close, last = [], -RESULT_WAIT['32x32'] - 1
    for i, x in enumerate(code):
        if x.mfma or before[i] != [i - 1]:
            last = i
        close.append(i - last <= RESULT_WAIT['32x32'])
    for i, x in enumerate(code):
        if x.mfma:
            count += 1
            operands = frozenset().union(*x.regs[1:])
            for w, gap in _writers_within(code, before, i, OPERAND_WAIT, lambda w: w.valu and w.writes & operands):
                out.append(f'{w.op} at {w.address:x} is {gap} wait states ahead of the {x.op} at {x.address:x}')
        elif x.touched and close[i]:
            for shape, wait in RESULT_WAIT.items():
                for w, gap in _writers_within(code, before, i, wait, lambda w: w.mfma and shape in w.op and w.regs[0] & x.touched):
                    out.append(f'{x.op} at {x.address:x} is {gap} wait states behind the {w.op} at {w.address:x}')
    assert count > 0
    return out


def test_checker_sees_a_short_distance():
    """The checker itself, on a listing written by hand: a loop whose last instruction writes a scale that the
    first one reads, and an accumulator that is read too early."""
    listing = '\n'.join([
        '\tv_mfma_scale_f32_16x16x128_f8f6f4 a[0:3], v[8:15], v[16:23], a[0:3], v2, v3 op_sel_hi:[0,0,0] // 000000001000: 00000000',
        '\ts_nop 7                                                    // 000000001010: BF800007',
        '\tv_accvgpr_read_b32 v30, a1                                 // 000000001014: 00000000',
        '\tv_lshrrev_b32_e32 v3, v4, v5                               // 00000000101C: 00000000',
        '\ts_waitcnt lgkmcnt(0)                                       // 000000001020: BF8CC07F',
        '\ts_cbranch_scc1 65528                                       // 000000001024: BF85FFF8 <dg_jit_kernel+0x0>',
        '\ts_endpgm                                                   // 000000001028: BF810000',
    ])
    found = violations(listing)
    assert len(found) == 1 and 'v_accvgpr_read_b32' in found[0], found     # (two states lie behind the shift)
    found = violations(listing.replace('s_waitcnt lgkmcnt(0)', 'v_mul_f32_e32 v3, v4, v5'))
    assert len(found) == 2 and any('v_mul' in f and '1 wait' in f for f in found), found
    assert violations(listing.replace('s_nop 7', 's_nop 15')) == []


FP8, FP8FP4, BF16 = _lib.DG_KIND_FP8_FP8, _lib.DG_KIND_FP8_FP4, _lib.DG_KIND_BF16
NORMAL, PSUM, MASKED = _lib.DG_GEMM_NORMAL, _lib.DG_GEMM_MGROUPED_PSUM, _lib.DG_GEMM_MASKED


@pytest.mark.parametrize('kind,gemm_type,m,n,k,alignment,fixed_k', [
    (FP8, NORMAL, 4096, 4096, 128, 256, True), (FP8, NORMAL, 1024, 2112, 384, 256, True), (FP8, NORMAL, 4096, 7168, 384, 256, True),
    (FP8, NORMAL, 1024, 2112, 2048, 256, True), (FP8FP4, NORMAL, 1024, 2112, 128, 256, True), (FP8, MASKED, 1024, 4096, 384, 256, True),
    (FP8, PSUM, 4096, 4096, 128, 128, True), (FP8FP4, PSUM, 4096, 4096, 384, 128, True),
    (FP8, PSUM, 4096, 4096, 384, 128, False), (BF16, NORMAL, 1024, 2112, 192, 256, True)])
def test_jit_wait_states(tmp_path, monkeypatch, kind, gemm_type, m, n, k, alignment, fixed_k):
    if not os.path.exists(OBJDUMP):
        pytest.skip('no llvm-objdump')
    monkeypatch.setenv('DG_JIT_CACHE_DIR', str(tmp_path))
    a = _args(m, n, k, gemm_type, _lib.DG_COMPILED_N | (_lib.DG_COMPILED_K if fixed_k else 0))
    a.kind, a.alignment, a.grouped_layout = kind, alignment, 0x600000
    lib = _lib.load()
    _lib.check(lib.dg_jit_compile(ctypes.byref(a)), lib)
    built = [f for f in os.listdir(tmp_path) if f.endswith('.hsaco')]
    assert len(built) == 1
    listing = subprocess.run([OBJDUMP, '-d', '--mcpu=gfx950', str(tmp_path / built[0])], capture_output=True, text=True,
                             check=True, timeout=120).stdout
    assert 'ds_read' in listing and 'v_mfma' in listing
    found = violations(listing)
    assert not found, (len(found), found[:8])


def test_ahead_of_time_wide_tiles(tmp_path):
    """The 384-row tiles, whose loops hold the scales' shifts in place without an asm of their own."""
    if not os.path.exists(OBJDUMP):
        pytest.skip('no llvm-objdump')
    fat = tmp_path / 'fatbin'
    subprocess.run([LLVM + 'llvm-objcopy', f'--dump-section=.hip_fatbin={fat}', str(_lib.library_path()), '/dev/null'],
                   check=True, timeout=60)
    checked = 0
    for i, part in enumerate(fat.read_bytes().split(b'__CLANG_OFFLOAD_BUNDLE__')[1:]):
        if b'quad_kernelILi384' not in part:
            continue
        bundle, obj = tmp_path / f'bundle{i}', tmp_path / f'obj{i}'
        bundle.write_bytes(b'__CLANG_OFFLOAD_BUNDLE__' + part)
        subprocess.run([LLVM + 'clang-offload-bundler', '--unbundle', '--type=o', '--targets=hipv4-amdgcn-amd-amdhsa--gfx950',
                        f'--input={bundle}', f'--output={obj}'], check=True, timeout=60)
        listing = subprocess.run([OBJDUMP, '-d', '--mcpu=gfx950', str(obj)], capture_output=True, text=True, check=True,
                                 timeout=120).stdout
        functions = re.split(r'^[0-9a-f]{16} <(.*)>:\n', listing, flags=re.M)[1:]
        for name, body in zip(functions[::2], functions[1::2]):
            if 'quad_kernelILi384' in name:
                found = violations(body)
                assert not found, (name, len(found), found[:8])
                checked += 1
    assert checked >= 6
