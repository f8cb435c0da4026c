"""Inline assembly tells the compiler of the registers that it writes by name: what is not named among the clobbers the compiler may hold a
value in."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'var_q_amd', 'csrc')


def test_registers_written_by_name_are_clobbers():
    seen = 0
    for path in sorted(glob.glob(os.path.join(CSRC, '*'))):
        if not path.endswith(('.hip', '.h', '.cpp')):
            continue
        text = re.sub(r'//[^\n]*', '', open(path).read())
        for m in re.finditer(r'\basm\s*(?:volatile)?\s*\((.*?)\)\s*;', text, re.S):
            body = m.group(1)
            strings = re.findall(r'"((?:[^"\\]|\\.)*)"', body)
            for reg in re.findall(r's_\w+\s+(m0|exec|vcc|s\d+|v\d+)\b', ' '.join(strings)):
                seen += 1
                assert reg in strings, f'{os.path.basename(path)}: {body.strip()} writes {reg}, which is not among its clobbers'
    assert seen == 3      # the copies of wide_attn.hip, one form for each of three lengths
