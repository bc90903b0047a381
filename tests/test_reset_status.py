"""A stream reset that fails on the GPU is reported.

The reset of a session is one launch per component (encoder caches, decoder state); a failure there
would let the next utterance run on the last one's state.  The host sources are compiled against a
device layer of stubs whose reset launch fails on demand.
"""
import os
import shutil
import subprocess

import pytest

from conftest import REPO

HOST = os.path.join(REPO, "nemo-c_amd", "csrc", "host")

COMPONENTS = r"""
#include "decoder.h"
#include "encoder.h"
#include "nemo_kernels.h"
#include <stdlib.h>
static int fail_reset, nomem;
struct gpu_buf { char b[64]; };
gpu_buf_t *gpu_buf_alloc(gpu_t *g, size_t n) { return nomem ? NULL : calloc(1, sizeof(gpu_buf_t)); }
void *gpu_buf_dptr(gpu_buf_t *b) { return b; }
void gpu_buf_free(gpu_buf_t *b) { free(b); }
void *gpu_host_alloc(gpu_t *g, size_t n) { return calloc(1, n); }
void gpu_host_free(void *p) { free(p); }
void gpu_graph_free(gpu_graph_t *p) {}
int gpu_cu_count(gpu_t *g) { return 0; }
int gpu_begin(gpu_t *g) { return 0; }
int gpu_end(gpu_t *g, char *e, size_t n) { return 0; }
int gpu_fail(gpu_t *g, const char *m) { return -1; }
int gpu_launch(gpu_t *g, const char *k, const void *a, size_t n, uint32_t x, uint32_t y, uint32_t z, uint32_t u, uint32_t v,
               uint32_t w) { return 0; }
int nk_stream_reset(gpu_t *g, const NkResetArgs *a) { return fail_reset ? -1 : 0; }
int main(void) {
    static model_t m;
    m.cfg = (model_cfg_t){ .n_layers = 2, .d_model = 64, .n_heads = 1, .head_dim = 64, .d_ff = 128, .subsampling = 8,
                           .sub_channels = 8, .conv_kernel = 9, .feat_in = 16, .prompt_hidden = 32, .pred_hidden = 32,
                           .joint_hidden = 32, .blank_id = 3, .att_left = 8 };
    decoder_t *d = decoder_create(&m);
    encoder_t *e = encoder_create(&m, 0);
    if (!d || !e || decoder_reset(d) || encoder_reset(e)) return 1;
    fail_reset = 1;
    if (!decoder_reset(d)) return 2;
    if (!encoder_reset(e)) return 3;
    if (decoder_create(&m)) return 4;
    fail_reset = 0;
    if (decoder_reset(d) || encoder_reset(e)) return 5;
    nomem = 1; /* buffers that were never allocated */
    encoder_t *f = encoder_create(&m, 0);
    if (!encoder_reset(f)) return 6;
    if (decoder_create(&m)) return 7;
    return 0;
}
"""

SESSION = r"""
#include "decoder.h"
#include "encoder.h"
#include "nemoasr.h"
#include "mel.h"
#include "resample.h"
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
static int fail_enc, fail_dec, steps;
static model_t model;
model_t *model_load(const char *d, char *e, size_t n) { return &model; }
void model_free(model_t *m) {}
int model_set_language(model_t *m, const char *l, char *e, size_t n) { return 0; }
int model_right_context_trained(const model_t *m, int r) { return 1; }
const char *gpu_last_error(gpu_t *g) { return "stub launch failed"; }
decoder_t *decoder_create(model_t *m) { return calloc(1, 8); }
void decoder_destroy(decoder_t *d) { free(d); }
int decoder_reset(decoder_t *d) { return fail_dec ? -1 : 0; }
void decoder_use_graphs(decoder_t *d, int on) {}
encoder_t *encoder_create(model_t *m, int r) { return calloc(1, 8); }
void encoder_destroy(encoder_t *e) { free(e); }
int encoder_reset(encoder_t *e) { return fail_enc ? -1 : 0; }
int encoder_chunk_mel(const encoder_t *e) { return 8; }
void encoder_set_dump(encoder_t *e, int on) {}
void encoder_use_graphs(encoder_t *e, int on) {}
void encoder_fuse(encoder_t *e, int on) {}
void encoder_chain(encoder_t *e, int on) {}
int encoder_chain_usable(const encoder_t *e) { return 0; }
void encoder_capture_first(encoder_t *e, int on) {}
void encoder_push(encoder_t *e, const float *x, size_t n) {}
int encoder_step(encoder_t *e, int f, enc_out_t *o, char *err, size_t n) { steps++; return 0; }
melfe_t *melfe_create(void) { return calloc(1, 8); }
void melfe_destroy(melfe_t *m) { free(m); }
void rsmp_destroy(rsmp_t *r) {}
size_t melfe_samples(const melfe_t *m) { return 0; }
void melfe_push(melfe_t *m, const float *x, size_t n, int f, const float **rows, size_t *k) { *rows = x; *k = 0; }
static int reset(nemoasr_t *s, int ms) {
    char err[256] = "";
    const int rc = nemoasr_reset(s, NULL, ms, err, sizeof err);
    if (rc && !strstr(err, "stub launch failed")) { printf("no reason: %s\n", err); exit(9); }
    return rc;
}
int main(void) {
    char err[256] = "";
    const float audio[160] = { 0 };
    nemoasr_t *s = nemoasr_open("x", NULL, 80, 16000, err, sizeof err);
    if (!s || reset(s, 80)) return 1;
    fail_enc = 1;
    if (!reset(s, 80)) return 2;
    steps = 0;
    free(nemoasr_feed(s, audio, 160, 1, err, sizeof err));
    if (steps) return 3; /* the half-reset stream takes no audio */
    if (!reset(s, 560)) return 4; /* preparing another chunk shape */
    if (nemoasr_prepare_latency(s, 1120, err, sizeof err) != -1) return 5;
    fail_enc = 0;
    if (nemoasr_prepare_latency(s, 1120, err, sizeof err)) return 6;
    fail_dec = 1;
    if (!reset(s, 80)) return 7;
    fail_dec = 0;
    if (reset(s, 560)) return 8;
    nemoasr_close(s);
    fail_enc = 1;
    return nemoasr_open("x", NULL, 80, 16000, err, sizeof err) ? 10 : 0;
}
"""


@pytest.mark.parametrize("name", ["components", "session"])
def test_failed_reset_is_reported(tmp_path, name):
    if not shutil.which("gcc"):
        pytest.skip("gcc not present")
    main, sources = (COMPONENTS, ["decoder.c", "encoder.c"]) if name == "components" else (SESSION, ["nemoasr.c"])
    src, exe = tmp_path / "main.c", tmp_path / name
    src.write_text(main)
    cc = ["gcc", "-std=c11", "-D_GNU_SOURCE", "-w", f"-I{HOST}", f"-I{REPO}/include", f"-I{HOST}/.."]
    objs = []
    for s in [str(src)] + [os.path.join(HOST, s) for s in sources]:
        objs.append(str(tmp_path / (os.path.basename(s) + ".o")))
        subprocess.run(cc + ["-c", s, "-o", objs[-1]], check=True)
    # what these runs do not call
    nm = subprocess.run(["nm", *objs], check=True, capture_output=True, text=True).stdout.split("\n")
    defined = {l.split()[2] for l in nm if len(l.split()) == 3}
    rest = sorted({l.split()[1] for l in nm if l.split()[:1] == ["U"]} - defined)
    rest = [f for f in rest if f.startswith(("gpu_", "nk_", "encoder_", "decoder_", "model_", "melfe_", "rsmp_", "piece_"))]
    other = tmp_path / "rest.c"
    other.write_text("#include <stdio.h>\n#include <stdlib.h>\n" +
                     "".join(f"int {f}() {{ puts(__func__); exit(99); }}\n" for f in rest))
    subprocess.run(["gcc", "-w", *objs, str(other), "-o", str(exe), "-lm"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout + r.stderr)
