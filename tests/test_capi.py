"""The C-ABI library: loads, exports what the header declares, validates arguments on the
host before anything is launched (CPU only; no kernel runs here)."""
import ctypes as C
import os
import re
import subprocess

import pytest

from deepstrix_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "dsx_moe.h")


def declared_functions():
    """name -> parameter count, parsed from the header's prototypes."""
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    text = re.sub(r"//[^\n]*", "", text)
    out = {}
    for m in re.finditer(r"\b(dsx_[a-z0-9_]+)\s*\(([^;{}]*?)\)\s*;", text, flags=re.S):
        name, args = m.group(1), m.group(2).strip()
        out[name] = 0 if args in ("", "void") else args.count(",") + 1
    return out


def test_header_is_plain_c():
    res = subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-fsyntax-only", "-x", "c", HEADER],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr


def test_library_exports_every_declared_symbol():
    decl = declared_functions()
    assert len(decl) >= 25
    raw = C.CDLL(capi.LIB_PATH)
    missing = [n for n in decl if not hasattr(raw, n)]
    assert not missing, f"declared in include/dsx_moe.h but not exported: {missing}"


def test_binding_table_matches_the_header():
    decl = declared_functions()
    assert set(decl) == set(capi.SIGNATURES), set(decl) ^ set(capi.SIGNATURES)
    for name, n in decl.items():
        assert len(capi.SIGNATURES[name][1]) == n, name


def test_abi_version_and_constants():
    text = open(HEADER).read()
    ver = int(re.search(r"#define\s+DSX_ABI_VERSION\s+(\d+)", text).group(1))
    assert capi.lib().dsx_abi_version() == ver
    for cname, val in [("DSX_FMT_Q8_0", capi.FMT_Q8_0), ("DSX_FMT_MXFP4", capi.FMT_MXFP4),
                       ("DSX_ERR_INVALID_ARG", capi.ERR_INVALID_ARG), ("DSX_ERR_SHAPE", capi.ERR_SHAPE),
                       ("DSX_ERR_UNSUPPORTED", capi.ERR_UNSUPPORTED), ("DSX_ERR_DEVICE", capi.ERR_DEVICE)]:
        m = re.search(rf"#define\s+{cname}\s+\(?(-?\d+)\)?", text)
        assert m and int(m.group(1)) == val, cname


def test_layer_desc_struct_matches_the_header_field_order():
    text = open(HEADER).read()
    body = re.search(r"typedef struct\s*\{((?:(?!typedef).)*?)\}\s*dsx_moe_layer_desc;", text, flags=re.S)
    assert body, "dsx_moe_layer_desc not found"
    src = re.sub(r"/\*.*?\*/", "", body.group(1), flags=re.S)
    names = []
    for stmt in src.split(";"):
        stmt = stmt.strip()
        if not stmt:
            continue
        for part in stmt.split(","):
            names.append(re.findall(r"[A-Za-z_][A-Za-z0-9_]*", part)[-1])
    assert names == [f[0] for f in capi.LayerDesc._fields_]


def _desc(**kw):
    d = capi.LayerDesc()
    d.hidden, d.inter, d.n_expert, d.n_used = 512, 256, 8, 2
    d.gate_fmt = d.up_fmt = d.down_fmt = capi.FMT_MXFP4
    d.gate = d.up = d.down = 0x1000  # never dereferenced by create()
    d.router_mode = capi.ROUTER_SIGMOID
    for k, v in kw.items():
        setattr(d, k, v)
    return d


def _create(d):
    h = C.c_void_p()
    rc = capi.lib().dsx_moe_layer_create(C.byref(d), C.byref(h))
    return rc, h


def test_layer_create_validates_before_anything_touches_a_device():
    l = capi.lib()
    rc, h = _create(_desc())
    assert rc == 0 and h.value
    assert l.dsx_moe_layer_workspace_bytes(h, 4) > l.dsx_moe_layer_workspace_bytes(h, 1) > 0
    l.dsx_moe_layer_destroy(h)

    cases = [
        (dict(gate=None), capi.ERR_INVALID_ARG),
        (dict(n_used=0), capi.ERR_INVALID_ARG),
        (dict(n_used=9), capi.ERR_INVALID_ARG),            # more picks than experts
        (dict(hidden=520), capi.ERR_SHAPE),                # not a multiple of 256
        (dict(inter=96), capi.ERR_SHAPE),                  # MXFP4 down needs inter % 256 == 0
        (dict(up_fmt=capi.FMT_Q8_0), capi.ERR_UNSUPPORTED),
        (dict(gate_fmt=12, up_fmt=12), capi.ERR_SHAPE),    # a format id with no layout
        (dict(sh_inter=256), capi.ERR_INVALID_ARG),        # shared expert without weights
        (dict(router_mode=3), capi.ERR_INVALID_ARG),
    ]
    for kw, code in cases:
        rc, h = _create(_desc(**kw))
        assert rc == code, (kw, rc)
        assert not h.value
        assert l.dsx_last_error(), kw
    with pytest.raises(capi.DsxError) as ei:
        capi.check(_create(_desc(hidden=520))[0])
    assert ei.value.code == capi.ERR_SHAPE and "hidden=520" in ei.value.message


def test_null_layer_handles_are_errors():
    l = capi.lib()
    assert l.dsx_moe_layer_set_profile_events(None, None, None, None) == capi.ERR_INVALID_ARG
    assert l.dsx_moe_layer_workspace_bytes(None, 1) == 0
    l.dsx_moe_layer_destroy(None)  # a no-op, like free(NULL)


def test_operators_refuse_bad_arguments_before_any_launch():
    """Validation comes first in every entry point: these calls return an error code without a
    device (pointers are fake; nothing is launched when the arguments are refused)."""
    l = capi.lib()
    p = 0x1000  # a non-null, 16-byte aligned stand-in
    bad = [
        l.dsx_router_topk(None, p, p, p, None, 0, 1, 1.0, 1e-20, 1, 0, 1, 1),          # n_expert = 0
        l.dsx_router_topk(None, p, p, p, None, 64, 6, 1.0, 1e-20, 1, 3, 1, 1),         # mode 3
        l.dsx_router_topk(None, p, p, p, None, 64, 6, 1.0, 1e-20, 1, 1, 7, 2),         # 64 % 7 != 0
        l.dsx_router_hash_select(None, p, p, p, p, p, 64, 0, 10, 1.5, 6e-5, 1),        # n_used = 0
        l.dsx_router_hash_select(None, p, p, p, None, p, 64, 6, 10, 1.5, 6e-5, 1),     # null table
        l.dsx_moe_hetsplit_select(None, p, p, p, 2, 1, 6, 64, 1),                      # mode 2
        l.dsx_moe_group_build(None, p, p, p, p, p, p, 4, 6, 64, 65),                   # chunk 65
        l.dsx_moe_group_build(None, p, p, p, p, p, p, 70000, 6, 64, 4),                # b >= 65536
        l.dsx_moe_gate_up_batch(None, capi.FMT_MXFP4, p, p, p, p, p, p, 8, 8, 6, 0.0, 24, 2),   # rows % 16
        l.dsx_moe_gate_up_batch(None, 12, p, p, p, p, p, p, 8, 8, 6, 0.0, 32, 2),               # format id
        l.dsx_moe_gate_up_chunked_rows(None, capi.FMT_MXFP4, p, p, p, p, p, p, p, p, p, p, 4, 8, 8, 6, 65,
                                       0.0, 32, 2),                                              # chunk 65
        l.dsx_moe_down_by_expert(None, capi.FMT_MXFP4, p, p, p, p, p, p, p, p, 4, 8, 292, 6, 0, 32, 1),  # chunk 0
        l.dsx_q8_0_weights_from_hf(None, p, p, None, capi.SRC_F8E4M3, 64, 64, 0, 0, 1),   # fp8 without scales
        l.dsx_q8_0_weights_from_hf(None, p, p, p, capi.SRC_F8E4M3, 64, 64, 3, 2, 1),      # grid does not tile
        l.dsx_q8_0_weights_from_hf(None, p, p, None, capi.SRC_F32, 64, 48, 0, 0, 1),      # cols % 32
        l.dsx_q8_0_repack_rows(None, p, p, 4, 2),                                          # in place
        l.dsx_mxfp4_repack_hf_to_v2(None, p, p, p, 4, 7),                                  # nb % 8
        l.dsx_rms_norm(None, p, p, None, 64, 1e-6, 1) if hasattr(l, "dsx_rms_norm") else -1,
    ]
    assert all(rc < 0 for rc in bad), bad
    assert l.dsx_last_error()


def _thresholds(hidden, inter, n_expert, n_used, gate_fmt=None, down_fmt=None):
    """Default thresholds of a layer of that shape (no device needed: creating a layer whose
    shared expert rides with the routed ones only records pointers and sizes)."""
    import ctypes as C
    l = capi.lib()
    d = capi.LayerDesc()
    d.hidden, d.inter, d.n_expert, d.n_used = hidden, inter, n_expert, n_used
    d.gate_fmt = d.up_fmt = capi.FMT_MXFP4 if gate_fmt is None else gate_fmt
    d.down_fmt = capi.FMT_MXFP4 if down_fmt is None else down_fmt
    d.gate = d.up = d.down = 0x1000
    d.gate_bpe = d.up_bpe = d.down_bpe = 1 << 20
    d.router_mode, d.n_group, d.topk_group = 1, 1, 1
    h = C.c_void_p()
    assert l.dsx_moe_layer_create(C.byref(d), C.byref(h)) == 0, l.dsx_last_error()
    v = (C.c_uint32 * 6)()
    assert l.dsx_moe_layer_get_tuning(h, C.byref(v)) == 0
    l.dsx_moe_layer_destroy(h)
    return dict(zip(("chunk", "gemm", "gemm_q8", "decode_max", "narrow", "share"), (int(x) for x in v)))


def test_default_thresholds_follow_the_picks_per_expert():
    """The crossovers measured on four shapes, as picks per expert (include/dsx_moe.h:
    dsx_moe_layer_set_tuning): every shape gets its token counts from the ratios, none inherits the
    DeepSeek-V3 shape's."""
    v3 = _thresholds(7168, 2048, 256, 8)
    # by-expert overtakes the decode launch at 13 .. 14 tokens, the GEMM the by-expert kernels at 96 .. 128
    assert (v3["narrow"], v3["share"]) == (1, 4)
    assert 13 <= v3["decode_max"] <= 14 and 97 <= v3["gemm"] <= 128
    # 128 experts, top-8, inter 1024: by-expert overtakes the decode launch between 12 and 16 tokens,
    # the GEMM the by-expert kernels between 48 and 64
    e128 = _thresholds(4096, 1024, 128, 8)
    assert 12 <= e128["decode_max"] <= 15 and 49 <= e128["gemm"] <= 64
    # 64 experts, top-6, small matrices: 4 .. 5 tokens and 64 .. 96 tokens
    e64 = _thresholds(2048, 1536, 64, 6)
    assert 4 <= e64["decode_max"] <= 5 and 65 <= e64["gemm"] <= 96
    # config 1 (all Q8_0): the int8 GEMM is ahead from 16 tokens on and far ahead at 24
    q8 = _thresholds(2048, 1408, 64, 6, capi.FMT_Q8_0, capi.FMT_Q8_0)
    assert 12 <= q8["gemm_q8"] <= 24
    # MXFP4 gate/up with a Q8_0 down matrix (config 5): the GEMMs are ahead from 64 tokens on
    mixed = _thresholds(7168, 2048, 256, 8, capi.FMT_MXFP4, capi.FMT_Q8_0)
    assert 49 <= mixed["gemm_q8"] <= 64


@pytest.mark.parametrize("shape,decode_max", [
    # (hidden, inter, experts, top), last token count at which the decode launch was measured no slower than the narrow tile
    ((7168, 2048, 256, 8), 7), ((7168, 2048, 256, 4), 15), ((7168, 2048, 192, 8), 6), ((7168, 2048, 160, 8), 6), ((7168, 2048, 160, 6), 8),
    ((7168, 2048, 128, 8), 5), ((7168, 2048, 64, 8), 2), ((7168, 2048, 64, 4), 5), ((7168, 2048, 32, 4), 2), ((6144, 4096, 16, 2), 2),
    ((6144, 4096, 32, 2), 5), ((6144, 2560, 160, 6), 7), ((4096, 14336, 8, 2), 1), ((5120, 1536, 160, 6), 9), ((4096, 1024, 128, 8), 5), ((2048, 1536, 64, 6), 3)])
def test_planar_layers_leave_the_decode_launch_where_it_is_slower(shape, decode_max):
    t = _thresholds(*shape, capi.FMT_MXFP4_PLANAR, capi.FMT_MXFP4_PLANAR)
    assert t["decode_max"] == decode_max and t["gemm"] * 11 // 16 <= decode_max + 1 and t["narrow"] == 14


def _workspace_bytes(T, hidden, inter, n_expert, n_used, gate_fmt, down_fmt):
    l = capi.lib()
    d = _desc(hidden=hidden, inter=inter, n_expert=n_expert, n_used=n_used, gate_fmt=gate_fmt, up_fmt=gate_fmt,
              down_fmt=down_fmt, sh_inter=inter, sh_gate_fmt=gate_fmt, sh_up_fmt=gate_fmt, sh_down_fmt=down_fmt,
              sh_gate=0x1000, sh_up=0x1000, sh_down=0x1000)
    rc, h = _create(d)
    assert rc == 0, l.dsx_last_error()
    n = l.dsx_moe_layer_workspace_bytes(h, T)
    l.dsx_moe_layer_destroy(h)
    return n


def test_workspaces_do_not_grow():
    """A caller may hold a buffer of a size that dsx_moe_layer_workspace_bytes has returned, and
    dsx_moe_layer_forward_noalloc serves what fits DSX_NOALLOC_SCRATCH_BYTES: a new table of a path
    goes into a region that is idle at that time, not behind the others."""
    M, Q = capi.FMT_MXFP4, capi.FMT_Q8_0
    v3 = (7168, 2048, 256, 8)
    assert [_workspace_bytes(T, *v3, M, M) for T in (1, 15, 16, 64)] == [533504, 7899136, 8424704, 31908864]
    assert _workspace_bytes(64, *v3, M, Q) == 31908864
    assert _workspace_bytes(512, 2048, 1408, 64, 6, Q, Q) == 80995584
    noalloc = int(re.search(r"#define\s+DSX_NOALLOC_SCRATCH_BYTES\s+\((\d+)u << 20\)", open(HEADER).read()).group(1)) << 20
    for T, *shape in [(114, 1024, 256, 128, 8), (79, 1024, 768, 128, 8), (15, *v3)]:   # the largest that fit
        assert _workspace_bytes(T, *shape, M, M) <= noalloc < _workspace_bytes(T + 1, *shape, M, M), shape


def _streaming(tuning=(0, 0, 0, 0), decode=0, **kw):
    """First and last token count on the streaming kernels, after set_tuning and set_decode."""
    l = capi.lib()
    rc, h = _create(_desc(**kw))
    assert rc == 0, l.dsx_last_error()
    assert l.dsx_moe_layer_set_tuning(h, *tuning) == 0 and l.dsx_moe_layer_set_decode(h, decode, 0) == 0
    v = (C.c_uint32 * 2)()
    assert l.dsx_moe_layer_get_streaming(h, C.byref(v)) == 0
    l.dsx_moe_layer_destroy(h)
    return tuple(int(x) for x in v)


def _sh(inter):
    """A shared expert of the routed shape."""
    return dict(sh_inter=inter, sh_gate_fmt=capi.FMT_MXFP4, sh_up_fmt=capi.FMT_MXFP4, sh_down_fmt=capi.FMT_MXFP4,
                sh_gate=0x1000, sh_up=0x1000, sh_down=0x1000)


_V3 = dict(hidden=7168, inter=2048, n_expert=256, n_used=8)


@pytest.mark.parametrize("shape,slower,faster", [
    # (hidden, inter, experts, top), token counts at which the older path was measured faster, and streaming (a shared expert
    # of the routed shape among the slots)
    ((7168, 2048, 256, 8), [2, 3], [4, 6, 9, 64]),
    ((7168, 2048, 256, 4), [4], [8, 9, 17]),
    ((4096, 1024, 256, 4), [8], [12, 14, 20]),
    ((4096, 1024, 128, 8), [4], [6, 8, 37]),
    ((5120, 1536, 160, 6), [6], [8, 9, 12]),
    ((4096, 1536, 128, 4), [6], [12, 14]),
    ((2048, 1536, 64, 6), [4], [10, 16, 28]),
    ((2048, 768, 128, 8), [8], [14, 20, 40]),
    ((1536, 1536, 64, 6), [8], [19, 28, 64])])
def test_streaming_begins_where_it_is_faster(shape, slower, faster):
    first, last = _streaming(**dict(zip(("hidden", "inter", "n_expert", "n_used"), shape)), **_sh(shape[1]))
    assert max(slower) < first <= min(faster) and max(faster) <= last, (first, last)


# (hidden, inter, experts, top): first token count with a shared expert alike, without one, with a Q8_0 one
FIRST_STREAMING = {
    (7168, 2048, 256, 8): (4, 6, 7), (7168, 2048, 256, 6): (6, 8, 10), (7168, 2048, 256, 4): (7, 12, 14), (7168, 2048, 256, 16): (3, 3, 7),
    (4096, 2048, 128, 8): (4, 4, 7), (4096, 2048, 64, 4): (7, 7, 7), (4096, 1024, 128, 8): (6, 7, 9), (5120, 1536, 160, 6): (8, 9, 9),
    (3072, 1024, 128, 8): (8, 8, 9), (2048, 1536, 64, 6): (8, 8, 9), (2048, 768, 128, 8): (14, 14, 14), (1024, 512, 128, 8): (36, 36, 36),
    (1024, 1024, 64, 6): (24, 24, 24), (7168, 2048, 64, 8): (4, 4, 7), (7168, 2048, 32, 4): (7, 7, 9), (6144, 4096, 16, 4): (7, 7, 9),
    (2048, 1792, 64, 6): (8, 8, 9), (3072, 1024, 32, 4): (12, 12, 12), (3072, 1024, 64, 6): (8, 8, 9)}


def first_streaming(shape, **sh):
    return _streaming(**dict(zip(("hidden", "inter", "n_expert", "n_used"), shape)), **sh)[0]


@pytest.mark.parametrize("shape", FIRST_STREAMING)
def test_few_tokens_stream_where_that_was_measured_faster(shape):
    assert (first_streaming(shape, **_sh(shape[1])), first_streaming(shape)) == FIRST_STREAMING[shape][:2]


@pytest.mark.gpu   # (a shared expert of another format has a stream of its own)
@pytest.mark.parametrize("shape", FIRST_STREAMING)
def test_few_tokens_stream_beside_a_q8_0_shared_expert_where_that_was_measured_faster(shape):
    Q = capi.FMT_Q8_0
    assert first_streaming(shape, **dict(_sh(shape[1]), sh_gate_fmt=Q, sh_up_fmt=Q, sh_down_fmt=Q)) == FIRST_STREAMING[shape][2]


def test_values_that_the_caller_sets_are_not_passed_over_by_streaming():
    assert _streaming(**_V3) == (6, 575)   # (where the decode launch is left: the range reported is the range taken)
    mixed = dict(_V3, down_fmt=capi.FMT_Q8_0)
    assert _streaming(**mixed) == (2, 895)
    for tuning in [(4, 0, 0, 0), (0, 112, 0, 0), (0, 0, 0, 1)]:   # (the values that are the defaults)
        assert _streaming(tuning, **_V3) == _streaming(tuning, **mixed) == (0, 0)
    assert _streaming((0, 0, 14, 0), **_V3) == (15, 575)
    assert _streaming((0, 0, 5, 0), **_V3) == (9, 575)
    for form in (2, 3, 4):
        assert _streaming(decode=form, **_V3) == (15, 575)
        assert _streaming(decode=form, **mixed) == (2, 895)   # (no decode path beside a Q8_0 down matrix)
    assert _streaming(decode=1, **_V3) == (6, 575)


def test_streaming_range_of_an_all_q8_0_layer_is_reported():
    Q = capi.FMT_Q8_0
    q8 = dict(hidden=2048, inter=1408, n_expert=64, n_used=6, gate_fmt=Q, up_fmt=Q, down_fmt=Q)
    first, last = _streaming(**q8)
    assert first == 2 and 15 <= last < 43   # (below 1.5 and 4 picks per expert)
    for tuning in [(4, 0, 0, 0), (0, 16, 0, 0)]:
        assert _streaming(tuning, **q8) == (0, 0)
    assert _streaming((0, 0, 8, 1), **q8) == (first, last)   # (values of MXFP4 paths)
    for odd in (dict(gate=0x1004), dict(down=0x1004), dict(up_bpe=12), dict(hidden=4224), dict(inter=4224)):
        assert _streaming(**{**q8, **odd}) == (0, 0), odd


@pytest.mark.parametrize("shape,last", [
    # (hidden, inter, experts, top), last token count: 1.5 picks per expert where the int8 GEMM was measured faster from there on, else 4
    ((2048, 1408, 64, 6), 42), ((1024, 512, 64, 4), 23), ((1024, 512, 128, 8), 23), ((512, 2048, 64, 4), 23),
    ((512, 4096, 32, 4), 11), ((1024, 512, 32, 4), 11), ((2048, 512, 32, 4), 11), ((2048, 768, 128, 8), 23),
    ((4096, 1024, 32, 4), 31), ((4096, 1024, 128, 8), 63), ((4096, 1536, 128, 8), 63), ((2560, 1792, 96, 4), 95), ((3072, 2048, 64, 4), 63)])
def test_all_q8_0_streaming_ends_where_it_is_slower(shape, last):
    Q = capi.FMT_Q8_0
    got = _streaming(**dict(zip(("hidden", "inter", "n_expert", "n_used"), shape)), gate_fmt=Q, up_fmt=Q, down_fmt=Q)
    assert got == (2, last)


@pytest.mark.parametrize("odd", [dict(gate=0x1004), dict(up=0x1004), dict(down=0x1004), dict(gate_bpe=12), dict(up_bpe=12),
                                 dict(down_bpe=12), dict(sh_gate=0x1004), dict(sh_up=0x1004), dict(sh_down=0x1004),
                                 dict(hidden=7424), dict(inter=7424, sh_inter=7424),
                                 dict(gate_fmt=capi.FMT_Q8_0, up_fmt=capi.FMT_Q8_0, sh_inter=0)])
def test_operands_that_the_streaming_kernels_do_not_take(odd):
    """Weights that are not 8-byte aligned, rows of more than 28 super-blocks, other formats."""
    sh = _sh(2048)
    assert _streaming(**dict(_V3, **sh)) == (4, 575)
    assert _streaming(**{**_V3, **sh, **odd}) == (0, 0)


def test_missing_library_is_an_import_error_not_a_fallback(monkeypatch):
    monkeypatch.setattr(capi, "_lib", None)
    monkeypatch.setattr(capi, "LIB_PATH", os.path.join(ROOT, "deepstrix_amd", "lib", "absent.so"))
    with pytest.raises(ImportError, match="no CPU fallback"):
        capi.lib()


def test_the_package_never_reaches_into_the_oracle():
    pkg = os.path.join(ROOT, "deepstrix_amd")
    offenders = []
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".hpp", ".inc", ".h")):
                text = open(os.path.join(dirpath, f), errors="replace").read()
                if re.search(r"\boracle\b|dsx_ref_|libdsx_oracle", text):
                    offenders.append(f)
    assert not offenders, offenders
