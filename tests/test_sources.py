"""Rules for the device sources that no compiler checks."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_load_in_inline_asm():
    """The compiler takes the output registers of an asm statement as written when it ends and as free where they are unused, so a load
    that is still on its way there overwrites what lives in them by then, an address among others."""
    sources = [f for d in ('dlblas_amd/csrc', 'bench_kernels') for f in glob.glob(os.path.join(ROOT, d, '*')) if f.endswith(('.h', '.hip', '.cpp'))]
    assert len(sources) > 10
    found = []
    for path in sources:
        text = open(path).read()
        for m in re.finditer(r'\basm\b\s*(?:volatile\s*)?\(', text):
            template = re.match(r'\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', text[m.end():])
            if template and re.search(r'\b(ds_read|ds_load|global_load|buffer_load|flat_load|scratch_load|s_load)', template[1]):
                found.append(f'{os.path.relpath(path, ROOT)}:{text[:m.start()].count(chr(10)) + 1}')
    assert not found, found
