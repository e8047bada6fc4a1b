"""What a layer and an encoder launch, seen on the host: their own sources linked against launch entries that only
write down what they were asked for, beside the kernels library for every question that a host function answers."""
import os
import subprocess

import pytest

from bytetransformer_amd import _lib, build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(build.CSRC, "host")
SOURCE = r"""
#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <vector>

#include "bytetransformer/bert_encoder.h"
#include "bytetransformer/bert_transformer.h"
using namespace bytetransformer;

static int slices = 0, asked = 0, live_by_size = 0;   // of FFN2; questions after them; products of known rows
struct Span {
  const char *begin, *end;
};
static Span partials, scratch;
static int prologues = 0, prologue_copies = 0, ln_copies = 0, norms_in_ffn1 = 0, qkv_starts = 0;
static bool norm_pays = false, only_ffn1_gains = false;   // what the kernels library would say on a GPU; whose copies pay
static std::vector<Span> others;   // what the LayerNorm behind the slices reads and writes, and what outlives it
static void take(const void *p, unsigned long long bytes) { others.push_back({(const char *)p, (const char *)p + bytes}); }
extern "C" {
int bt_layer_prologue(const void *, int, int, int, int *, int *, int *, int *, void *, int, int, int copies, const void *const *,
                      void *const *, const int *, const int *, int, const void *const *, const unsigned long long *, void *) {
  ++prologues, prologue_copies += copies;
  return 0;
}
int bt_gemm_qkv_bias_split(const void *, const int *, const void *, const void *, void *, const int *, int, int, int, int, int, void *) { return 0; }
int bt_gemm_qkv_bias_split_mask_rows(const void *, const void *, int, int, int, const void *, const void *, void *, int *, int *,
                                     int *, int, int, int, int, void *) {
  ++qkv_starts;
  return 0;
}
int bt_attention_grouped(const void *, void *, const int *, const int *, const void *, const void *, int, int, int, int, int,
                         float, int, const void *const *, const unsigned long long *, int, const int *slots, const void *list, void *) {
  if (slots) take(slots, 256 * sizeof(int));
  if (list) take(list, 16);
  return 0;
}
int bt_mask_prefix_slots(const void *, int, int, int, const int *, int *, void *) { return 0; }
int bt_add_bias_residual_layernorm(void *, const void *, const int *, const void *, const void *, const void *, int, const int *,
                                   int, int, float, void *) { return 0; }
int bt_add_bias_residual_layernorm_copy(void *, const void *, const int *, const void *, const void *, const void *, int,
                                        const int *, int, int, float, int copies, const void *const *, void *const *, const int *,
                                        const int *, void *) {
  ln_copies += copies;
  return 0;
}
int bt_add_bias_residual_layernorm_restore(const void *, const void *, const void *, const void *, const void *, int, void *,
                                           const int *, const int *, int, int, int, float, void *) { return 0; }
int bt_splitk_layernorm(const void *sums, int splits, const void *residual, const int *, const void *, const void *, const void *,
                        int, void *dst, const int *offsets, const int *live, int, int, int rows, int n, float, void *) {
  partials = {(const char *)sums, (const char *)sums + 4ull * splits * rows * n};
  take(residual, 2ull * rows * n);
  take(dst, 2ull * rows * n);
  if (offsets) take(offsets, 4);
  if (live) take(live, 4);
  return 0;
}
int bt_gemm(const void *, const void *, void *, const int *live, int, int, int n, int k, int, void *) {
  if (k > n) slices = 1;
  live_by_size += live == nullptr;
  return 0;
}
int bt_gemm_bias_gelu(const void *, const void *, const void *, void *, const int *live, int, int, int, int, int, void *) {
  live_by_size += live == nullptr;
  return 0;
}
int bt_layernorm_gemm_bias_gelu(const void *, const void *, const int *, const void *, const void *, const void *, void *,
                                const void *, const void *, void *, const int *, int, int all_live, int, int, int, float, void *) {
  live_by_size += all_live;
  ++norms_in_ffn1;
  return 0;
}
int bt_layernorm_gemm_bias_gelu_pays(int rows_cap, int all_live, int n, int k, int weight_kn) {
  if (norm_pays) return rows_cap <= 111;
  return ((int (*)(int, int, int, int, int))dlsym(RTLD_NEXT, "bt_layernorm_gemm_bias_gelu_pays"))(rows_cap, all_live, n, k, weight_kn);
}
float bt_gemm_prepack_gain_us(long long rows, int n, int k, int epilogue) {
  if (only_ffn1_gains) return epilogue == BT_EPILOGUE_BIAS_GELU ? 5.f : 0.f;
  return ((float (*)(long long, int, int, int))dlsym(RTLD_NEXT, "bt_gemm_prepack_gain_us"))(rows, n, k, epilogue);
}
int bt_gemm_splitk_rows(const void *a, const void *, void *, int splits, const int *live, int rows, int, int, int k, int, void *) {
  slices = splits;
  take(a, 2ull * rows * k);
  if (live) take(live, 4);
  live_by_size += live == nullptr;
  return 0;
}
int bt_gemm_splitk_slices(int rows_cap, int all_live, int n, int k, int most) {
  ++asked;
  return ((int (*)(int, int, int, int, int))dlsym(RTLD_NEXT, "bt_gemm_splitk_slices"))(rows_cap, all_live, n, k, most);
}
}

// argv: layer|encoder  heads  batch  seq_len  live rows that the caller vouches for (-1: no offsets, -2: padded rows)
// [batch and seq_len that the scratch is for]
// or: plan  heads  batch  seq_len  live  (1: the first LayerNorm's launch may be FFN1's)  (1: only FFN1's copy pays)
// (1: the LayerNorm's launch may carry copies): launches of a layer, and what its plan says of them
static int plan_and_launches(char **argv) {
  const int heads = std::atoi(argv[2]), batch = std::atoi(argv[3]), seq = std::atoi(argv[4]), live = std::atoi(argv[5]);
  norm_pays = std::atoi(argv[6]) != 0, only_ffn1_gains = std::atoi(argv[7]) != 0;
  bt_set_option("ln_weight_copy", std::atoi(argv[8]));
  bt_set_option("layer_prepack", only_ffn1_gains ? -1 : 1);
  static char some[4096];
  const __half *t = (const __half *)some;
  BertTransformerParam<OperationType::HALF> w;
  w.attention_param.attr_bias_QKV = t;
  w.attr_kernel_QKV = w.attr_output_kernel = w.inter_kernel = w.output_kernel = t;
  BertTransformer<OperationType::HALF> layer(batch, heads, 64, seq, true, live != -2);
  layer.initialize(w);
  BertTransformerInferParam<__half> ip{t, t, (__half *)some, some, batch, seq, nullptr, nullptr};
  ET_Param offsets{(int *)some, (int *)some, live};
  if (live >= 0) ip.offsets = &offsets;
  const LayerPlan lp = layer.plan(batch, seq, live >= 0, 0, live > 0 ? live : 0);
  layer.infer(ip);
  int copies = 0, by_ln = 0;
  for (int i = 0; i < 4; ++i) copies += lp.copy[i], by_ln += lp.ln_copy[i];
  std::printf("%d %d %d %d %d %d %d %d %d\n", prologues, prologue_copies, copies, lp.copies, ln_copies, by_ln, norms_in_ffn1,
              lp.norm_in_ffn1, qkv_starts == lp.starts_with_qkv);
  return 0;
}

int main(int argc, char **argv) {
  if (argv[1][0] == 'p') return plan_and_launches(argv);
  const int heads = std::atoi(argv[2]), batch = std::atoi(argv[3]), seq = std::atoi(argv[4]), live = std::atoi(argv[5]);
  const int most = argc > 7 ? std::atoi(argv[6]) : batch, longest = argc > 7 ? std::atoi(argv[7]) : seq;
  const bool packed = live != -2;
  static char some[4096];
  const __half *t = (const __half *)some;
  BertTransformerParam<OperationType::HALF> w;
  w.attention_param.attr_bias_QKV = t;
  w.attr_kernel_QKV = w.attr_output_kernel = w.inter_kernel = w.output_kernel = t;
  if (argv[1][0] == 'l') {
    BertTransformer<OperationType::HALF> layer(most, heads, 64, longest, true, packed);
    layer.initialize(w);
    scratch = {some, some + layer.cal_bufsize()};
    BertTransformerInferParam<__half> ip{t, t, (__half *)some, some, batch, seq, nullptr, nullptr};
    ET_Param offsets{(int *)some, (int *)some, live};
    if (live >= 0) ip.offsets = &offsets;
    layer.infer(ip);
  } else {
    BertEncoder<OperationType::HALF> encoder(most, heads, 64, longest, true, packed);
    encoder.initialize(std::vector<BertTransformerParam<OperationType::HALF>>(12, w));
    scratch = {some, some + encoder.cal_bufsize()};
    BertEncoderInferParam<__half> ip{};
    ip.input_tensor = ip.atten_mask = t, ip.transformer_output = (__half *)some, ip.buf = some;
    ip.batch_size = batch, ip.seq_len = seq;
    encoder.infer(ip);
  }
  bool apart = partials.begin == partials.end || (partials.begin >= scratch.begin && partials.end <= scratch.end);
  for (const Span &o : others) apart = apart && (o.begin >= partials.end || o.end <= partials.begin);
  std::printf("%d %d %d %d\n", slices, live_by_size, asked, apart);
}
"""


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("launches")
    source, program = str(tmp / "launches.cc"), str(tmp / "launches")
    with open(source, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++"] + build.HOST_FLAGS +
                   ["-I", os.path.join(ROOT, "include"), "-I", HOST, "-I", os.path.join(build.ROCM, "include"), source] +
                   [os.path.join(HOST, f) for f in ("bert_transformer.cc", "bert_encoder.cc", "attention.cc")] +
                   ["-L", build.LIB, "-lbt_hip", "-L", os.path.join(build.ROCM, "lib"), "-lamdhip64", "-ldl",
                    "-Wl,-rpath," + build.LIB, "-Wl,-rpath," + os.path.join(build.ROCM, "lib"), "-o", program], check=True)
    env = {k: v for k, v in os.environ.items() if k != "BT_SPLITK"}

    def run(*args):
        out = subprocess.run([program] + [str(a) for a in args], check=True, stdout=subprocess.PIPE, text=True, env=env)
        return tuple(int(v) for v in out.stdout.split())
    return run


# live rows of hidden 768 -> slices: what the sizes give where every row is live (a padded batch of 900 rows gets 2,
# one of 1050 gets 2, of 2400 three)
@pytest.mark.parametrize("live,slices", [(32, 4), (900, 4), (1050, 4), (1500, 3), (2100, 2), (2400, 2), (3400, 1), (8192, 1)])
def test_offsets_with_their_count(launches, live, slices):
    got, live_by_size, _, _ = launches("layer", 12, 16, 512, live)
    assert got == slices == _lib.kernel_lib().bt_gemm_splitk_slices(live, 1, 768, 3072, 16)
    assert live_by_size == 3


@pytest.mark.parametrize("batch,seq_len", [(16, 512), (4, 96), (7, 217), (8, 300)])
def test_offsets_without_their_count(launches, batch, seq_len):
    """A caller that does not know the count gets the slices of one that passes no offsets."""
    own = launches("layer", 12, batch, seq_len, -1)[:3]
    assert launches("layer", 12, batch, seq_len, 0)[:3] == own
    assert own[1] == 0


def test_padded_rows_are_all_live(launches):
    got = launches("layer", 12, 2, 200, -1)
    assert got[0] == _lib.kernel_lib().bt_gemm_splitk_slices(400, 1, 768, 3072, 16)


@pytest.mark.parametrize("batch,seq_len", [(1, 32), (4, 96), (16, 512)])
def test_an_encoder_asks_once_for_its_slices(launches, batch, seq_len):
    slices, _, asked, _ = launches("encoder", 12, batch, seq_len, -1)
    assert asked == 1 and slices == launches("layer", 12, batch, seq_len, -1)[0]


@pytest.mark.parametrize("kind", ["layer", "encoder"])
@pytest.mark.parametrize("heads", [8, 12, 16])
def test_partial_sums_lie_apart(launches, kind, heads):
    """FFN2's partial sums lie in the scratch and touch nothing that their LayerNorm reads or writes, nor what a later
    layer reads again: sizes around those where the slices change, packed and padded rows, exact counts, scratch for
    just these sizes and for more."""
    seen = set()
    for batch, seq_len in ((1, 1), (1, 32), (3, 33), (4, 96), (1, 700), (7, 217), (8, 250), (8, 300), (8, 313), (5, 640), (16, 512)):
        for live in (-1, -2) + ((batch * seq_len, batch * seq_len * 3 // 5) if kind == "layer" else ()):
            for room in ((), (batch + 1, seq_len), (2 * batch, seq_len + 100)):
                slices, _, _, apart = launches(kind, heads, batch, seq_len, live, *room)
                assert apart, (batch, seq_len, live, room, slices)
                seen.add(slices)
    assert len(seen) >= 3, seen


@pytest.mark.parametrize("live", [-1, -2, 30])   # its own offsets, padded rows, offsets with their count
@pytest.mark.parametrize("only_ffn1_gains", [0, 1])
@pytest.mark.parametrize("ln_weight_copy", [0, 1])
@pytest.mark.parametrize("norm_pays", [0, 1])
@pytest.mark.parametrize("batch,seq_len", [(1, 32), (3, 14), (3, 60)])   # (up to two sequences: padded rows)
def test_the_plan_is_what_is_launched(launches, batch, seq_len, norm_pays, ln_weight_copy, only_ffn1_gains, live):
    """Copies and where they are made, whether the first LayerNorm is in FFN1's launch, and whether the layer starts with the
    QKV product: with the LayerNorm in FFN1's launch there is no copy for FFN1, and no prologue that only it would need."""
    prologues, made, planned, count, ln_made, ln_planned, norms, norm_planned, starts = launches(
        "plan", 12, batch, seq_len, live, norm_pays, only_ffn1_gains, ln_weight_copy)
    assert (made, ln_made, norms) == (planned, ln_planned, norm_planned) and count == planned and starts
    rows = live if live > 0 and batch > 2 else batch * seq_len
    assert norms == (norm_pays and rows <= 111)
    if norms:
        assert ln_made == 0 and made <= 3 and not (only_ffn1_gains and made)
        if only_ffn1_gains and live == -1:
            assert prologues == 0
