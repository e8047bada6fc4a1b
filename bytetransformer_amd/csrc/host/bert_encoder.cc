// BertEncoder<OpType>::infer - a stack of encoder layers over the C ABI with the
// hidden state kept packed between layers.  Per layer the operation order and
// residual choices are those of one reference layer (bert_transformer.cu:28-130);
// the compress / restore pair of every inner layer is dropped.
#include "bytetransformer/bert_encoder.h"

namespace bytetransformer {

template <OperationType OpType>
void BertEncoder<OpType>::prepack(void *prepacked, hipStream_t stream) const {
  if (OpType == OperationType::FP32) return;   // float weights are consumed as stored
  if (!prepacked) throw std::runtime_error("[BT][ERROR] BertEncoder::prepack: null destination");
  const int hidden = head_num_ * size_per_head_, inter = hidden * intermediate_size_;
  DataType_ *dst = (DataType_ *)prepacked;
  for (const auto &l : layers_) {
    DataType_ *wt_qkv = dst, *wt_proj = wt_qkv + (size_t)3 * hidden * hidden;
    DataType_ *wt_inter = wt_proj + (size_t)hidden * hidden, *wt_out = wt_inter + (size_t)hidden * inter;
    const void *src[4] = {l.attr_kernel_QKV, l.attr_output_kernel, l.inter_kernel, l.output_kernel};
    void *out[4] = {wt_qkv, wt_proj, wt_inter, wt_out};
    const int ks[4] = {hidden, hidden, hidden, inter};
    const int ns[4] = {3 * hidden, hidden, inter, hidden};
    check_bt_error(bt_transpose_weights(4, src, out, ks, ns, stream));
    dst += layer_weight_elems();
  }
}

template <OperationType OpType>
void BertEncoder<OpType>::infer(BertEncoderInferParam<DataType_> ip) {
  if (layers_.empty()) throw std::runtime_error("[BT][ERROR] BertEncoder: initialize() first");
  if (!ip.input_tensor || !ip.atten_mask || !ip.transformer_output || !ip.buf)
    throw std::runtime_error("[BT][ERROR] BertEncoder: null input/mask/output/buf pointer");
  const int batch_size = ip.batch_size, seq_len = ip.seq_len;
  if (batch_size <= 0 || seq_len <= 0 || batch_size > max_batch_size_ || seq_len > max_seq_len_)
    throw std::runtime_error(
        "[BT][ERROR] BertEncoder: batch_size/seq_len outside the constructed maximum");
  hipStream_t stream = ip.stream;

  const int hidden = head_num_ * size_per_head_, inter = hidden * intermediate_size_;
  const int rows = batch_size * seq_len;
  if (OpType == OperationType::HALF && hidden % 64 != 0)
    throw std::runtime_error("[BT][ERROR] BertEncoder: fp16 layers need head_num * size_per_head "
                             "to be a multiple of 64, got " + std::to_string(hidden));
  const size_t tensor = (size_t)rows * hidden;
  const unsigned long long max_rows = (unsigned long long)max_batch_size_ * max_seq_len_;
  const unsigned long long max_tensor = max_rows * hidden;

  uint8_t *base = (uint8_t *)ip.buf;
  unsigned long long off = 0;
  ET_Param et_param;
  et_param.word_idx = (int *)(base + off);
  et_param.batch_idx = et_param.word_idx + max_rows;
  et_param.valid_word_num = rows;
  int *seq_order = et_param.batch_idx + max_batch_size_ + 1;
  int *mask_slots = seq_order + max_batch_size_;       // int[256], padded path only
  off += align_up((max_rows * 2 + 2 * (unsigned long long)max_batch_size_ + 2 + 256) * sizeof(int),
                  256);
  DataType_ *inter_matmul_buf = (DataType_ *)(base + off);
  DataType_ *attr_matmul_buf = inter_matmul_buf + intermediate_size_ * max_tensor;   // projection, then LN1 in place
  DataType_ *hidden_buf = attr_matmul_buf + max_tensor;   // FFN2 out, then LN2 in place = next input
  // (what FFN2 leaves dead lies next to the split-k area: together they are what its partial sums may use)
  DataType_ *qkv_buf = hidden_buf + max_tensor;
  DataType_ *attr_out_buf = qkv_buf + 3 * tensor;
  off += align_up((6 + intermediate_size_) * max_tensor * sizeof(DataType_), 256);
  float *partials = (float *)qkv_buf;
  const unsigned long long splitk_bytes = splitk_scratch_bytes(max_rows, (unsigned long long)hidden);
  const unsigned long long partials_bytes = (base + off + splitk_bytes) - (uint8_t *)qkv_buf;
  off += align_up(splitk_bytes, 256);
  // the streaming attention's balanced work list: built once per forward beside the offsets
  void *work_list = nullptr;
  if (OpType == OperationType::HALF && size_per_head_ == 64 &&
      !attention_layer_->uses_short_kernel(seq_len) &&
      bt_attention_worklist_bytes(batch_size, seq_len, head_num_) > 0)
    work_list = base + off;

  // padded rows: the fp16 streaming attention applies the mask tensor unless one pass
  // over it (once for all layers) finds the plain prefix mask of the lengths
  const bool check_mask = !is_remove_padding_ && OpType == OperationType::HALF &&
                          size_per_head_ == 64;
  // offsets and that verdict in one launch, once per forward
  check_bt_error(bt_layer_prologue(ip.atten_mask, Traits_::dtype, batch_size, seq_len,
                                   et_param.batch_idx, et_param.word_idx, seq_order,
                                   check_mask ? mask_slots : nullptr, work_list, head_num_,
                                   is_remove_padding_ ? 0 : 1, 0, nullptr, nullptr, nullptr,
                                   nullptr, 0, nullptr, nullptr, stream));
  const int *valid_rows = is_remove_padding_ ? et_param.batch_idx + batch_size : nullptr;
  const int rows_hint = rows_to_plan_for(ip.valid_rows_hint, is_remove_padding_, batch_size, rows);
  const int L = (int)layers_.size();
  // few rows, long k: FFN2 as split-k partial sums that the last LayerNorm folds in (the same in every layer)
  const int splits =
      OpType == OperationType::HALF ? ffn2_slices(rows, valid_rows == nullptr, hidden, inter, partials_bytes) : 1;
  // few rows: the first LayerNorm in FFN1's launch, which reads the projection from where Q was
  const bool norm_in_ffn1 = OpType == OperationType::HALF && !use_fp32_ &&
                            bt_layernorm_gemm_bias_gelu_pays(rows, valid_rows == nullptr, inter, hidden, ip.prepacked ? 0 : 1);
  // float: weights split afresh in every layer where the rows are worth it
  const bool f32_split = OpType == OperationType::FP32 && f32_splits_operands(rows, !is_remove_padding_, hidden, inter);
  uint8_t *split_at = base + off + align_up(attention_layer_->work_list_capacity(), 256);
  void *w_pairs[4] = {split_at, split_at + 12ull * hidden * hidden, split_at + 16ull * hidden * hidden,
                      split_at + 16ull * hidden * hidden + 4ull * hidden * inter};
  const F32SplitScratch sp(split_at + align_up(layer_weight_elems() * sizeof(float), 256), max_rows, hidden, inter);

  for (int l = 0; l < L; ++l) {
    const auto &w = layers_[l];
    // layer 0 reads the caller's padded input (valid token t at row word_idx[t] when
    // packing), every later layer the packed hidden state
    const DataType_ *x = l == 0 ? ip.input_tensor : hidden_buf;
    const int *gather = (l == 0 && is_remove_padding_) ? et_param.word_idx : nullptr;

    const bool last = l == L - 1;
    // the last layer of the padded path writes straight into the caller's output
    DataType_ *ffn2_out = (last && !is_remove_padding_) ? ip.transformer_output : hidden_buf;
    attention_layer_->initialize(w.attention_param);

    if constexpr (OpType == OperationType::FP32) {
      // (the input's pairs lie in FFN1's area until that is written)
      if (f32_split) {
        const void *ws[4] = {w.attr_kernel_QKV, w.attr_output_kernel, w.inter_kernel, w.output_kernel};
        const int ks[4] = {hidden, hidden, hidden, inter}, ns[4] = {3 * hidden, hidden, inter, hidden};
        check_bt_error(bt_split_f32_layer(4, ws, w_pairs, sp.w_exps, ks, ns, 2, w.inter_bias, sp.bounds, x, inter_matmul_buf,
                                          sp.x_exps, gather, valid_rows, rows, hidden, 1, stream));
        const bt_f32_split_more qkv{0, nullptr, nullptr, w.attr_kernel_QKV, x, gather, ip.valid_rows_hint};
        check_bt_error(bt_gemm_f32_split_with(inter_matmul_buf, sp.x_exps, w_pairs[0], sp.w_exps[0],
                                              w.attention_param.attr_bias_QKV, qkv_buf, nullptr, valid_rows, rows, 3 * hidden,
                                              hidden, &qkv, stream));
      } else {
        check_bt_error(bt_gemm_f32(x, gather, w.attr_kernel_QKV, w.attention_param.attr_bias_QKV,
                                   qkv_buf, 0, valid_rows, rows, rows_hint, 3 * hidden, hidden, stream));
      }
      struct AttentionInferParam<DataType_> att {
        qkv_buf, ip.atten_mask, attr_out_buf, nullptr, batch_size, seq_len, nullptr, stream,
            et_param
      };
      att.attention_bias = ip.attention_bias;
      att.seq_order = seq_order;
      attention_layer_->infer(att);
      if (f32_split) {
        // (Q, K, V are dead: the attention's pairs take the first tensor's place, the LayerNorm's the second's)
        DataType_ *att_pairs = qkv_buf, *ln_pairs = qkv_buf + tensor;
        const bt_f32_split_more proj{0, nullptr, nullptr, w.attr_output_kernel, attr_out_buf, nullptr, ip.valid_rows_hint},
            ffn1{0, sp.raw, nullptr, w.inter_kernel, attr_matmul_buf, nullptr, ip.valid_rows_hint},
            ffn2{0, nullptr, sp.raw, w.output_kernel, nullptr, nullptr, ip.valid_rows_hint};
        check_bt_error(bt_split_f32_layer(0, nullptr, nullptr, nullptr, nullptr, nullptr, -1, nullptr, nullptr, attr_out_buf,
                                          att_pairs, sp.att_exps, nullptr, valid_rows, rows, hidden, 1, stream));
        check_bt_error(bt_gemm_f32_split_with(att_pairs, sp.att_exps, w_pairs[1], sp.w_exps[1], nullptr, attr_matmul_buf, nullptr,
                                              valid_rows, rows, hidden, hidden, &proj, stream));
        check_bt_error(bt_add_bias_residual_layernorm_f32_split_layer(
            attr_matmul_buf, x, gather, w.attr_output_bias, w.attr_output_layernorm_gamma, w.attr_output_layernorm_beta,
            valid_rows, rows, hidden, layernorm_eps, ln_pairs, sp.ln_exps, sp.gelu_exps, sp.bounds, sp.bound_count, sp.raw, inter,
            stream));
        check_bt_error(bt_gemm_f32_split_with(ln_pairs, sp.ln_exps, w_pairs[2], sp.w_exps[2], w.inter_bias, inter_matmul_buf,
                                              sp.gelu_exps, valid_rows, rows, inter, hidden, &ffn1, stream));
        check_bt_error(bt_gemm_f32_split_with(inter_matmul_buf, sp.gelu_exps, w_pairs[3], sp.w_exps[3], nullptr, ffn2_out, nullptr,
                                              valid_rows, rows, hidden, inter, &ffn2, stream));
      } else {
        check_bt_error(bt_gemm_f32(attr_out_buf, nullptr, w.attr_output_kernel, nullptr,
                                   attr_matmul_buf, 0, valid_rows, rows, rows_hint, hidden, hidden, stream));
        check_bt_error(bt_add_bias_residual_layernorm_f32(
            attr_matmul_buf, x, gather, w.attr_output_bias, w.attr_output_layernorm_gamma,
            w.attr_output_layernorm_beta, valid_rows, rows, hidden, layernorm_eps, stream));
        check_bt_error(bt_gemm_f32(attr_matmul_buf, nullptr, w.inter_kernel, w.inter_bias,
                                   inter_matmul_buf, 1, valid_rows, rows, rows_hint, inter, hidden, stream));
        check_bt_error(bt_gemm_f32(inter_matmul_buf, nullptr, w.output_kernel, nullptr, ffn2_out, 0,
                                   valid_rows, rows, rows_hint, hidden, inter, stream));
      }
      if (last && is_remove_padding_)
        check_bt_error(bt_add_bias_residual_layernorm_restore_f32(
            ffn2_out, attr_matmul_buf, w.output_bias, w.output_layernorm_gamma,
            w.output_layernorm_beta, ip.transformer_output, et_param.batch_idx, batch_size,
            seq_len, hidden, layernorm_eps, stream));
      else
        check_bt_error(bt_add_bias_residual_layernorm_f32(
            ffn2_out, attr_matmul_buf, nullptr, w.output_bias, w.output_layernorm_gamma,
            w.output_layernorm_beta, valid_rows, rows, hidden, layernorm_eps, stream));
      continue;
    }

    // pre-packed copies made when the encoder was created (its weights are private and
    // immutable), else the [k, n] weights as they are stored
    const int weight_kn = ip.prepacked ? 0 : 1;
    const DataType_ *wt_qkv = w.attr_kernel_QKV, *wt_proj = w.attr_output_kernel,
                    *wt_inter = w.inter_kernel, *wt_out = w.output_kernel;
    if (ip.prepacked) {
      wt_qkv = (const DataType_ *)ip.prepacked + (size_t)l * layer_weight_elems();
      wt_proj = wt_qkv + (size_t)3 * hidden * hidden;
      wt_inter = wt_proj + (size_t)hidden * hidden;
      wt_out = wt_inter + (size_t)hidden * inter;
    }

    check_bt_error(bt_gemm_qkv_bias_split(x, gather, wt_qkv, w.attention_param.attr_bias_QKV,
                                          qkv_buf, valid_rows, rows, rows_hint, head_num_,
                                          size_per_head_, weight_kn, stream));

    struct AttentionInferParam<DataType_> att {
      qkv_buf, ip.atten_mask, attr_out_buf, nullptr, batch_size, seq_len, nullptr, stream, et_param
    };
    att.attention_bias = ip.attention_bias;
    att.seq_order = seq_order;
    if (check_mask) att.mask_prefix_slots = mask_slots;
    att.work_list = work_list;
    // warm the caches with what follows: the rest of this layer's weights and the next layer's QKV matrix
    const void *next[4] = {wt_proj, wt_inter, wt_out, nullptr};
    if (l + 1 < L) next[3] = ip.prepacked ? (const void *)(wt_out + (size_t)hidden * inter) : layers_[l + 1].attr_kernel_QKV;
    const int next_k[4] = {hidden, hidden, inter, hidden}, next_n[4] = {hidden, inter, hidden, 3 * hidden};
    att.prefetch_count = l + 1 < L ? 4 : 3;
    for (int i = 0; i < att.prefetch_count; ++i) {
      att.prefetch[i] = next[i];
      att.prefetch_bytes[i] = prefetch_weight(next_k[i], next_n[i], weight_kn, i == 2 ? splits : 1, valid_rows ? rows * 3LL / 5 : rows);
    }
    attention_layer_->infer(att);

    check_bt_error(bt_gemm(attr_out_buf, wt_proj, norm_in_ffn1 ? qkv_buf : attr_matmul_buf, valid_rows, rows, rows_hint,
                           hidden, hidden, weight_kn, stream));
    if (norm_in_ffn1) {
      check_bt_error(bt_layernorm_gemm_bias_gelu(
          qkv_buf, x, gather, w.attr_output_bias, w.attr_output_layernorm_gamma, w.attr_output_layernorm_beta,
          attr_matmul_buf, wt_inter, w.inter_bias, inter_matmul_buf, valid_rows, rows, valid_rows == nullptr, inter, hidden,
          weight_kn, layernorm_eps, stream));
    } else {
      check_bt_error(bt_add_bias_residual_layernorm(
          attr_matmul_buf, x, gather, w.attr_output_bias, w.attr_output_layernorm_gamma,
          w.attr_output_layernorm_beta, use_fp32_ ? 1 : 0, valid_rows, rows, hidden, layernorm_eps,
          stream));
      check_bt_error(bt_gemm_bias_gelu(attr_matmul_buf, wt_inter, w.inter_bias, inter_matmul_buf,
                                       valid_rows, rows, rows_hint, inter, hidden, weight_kn,
                                       stream));
    }

    if (splits > 1) {
      const bool restore = last && is_remove_padding_;
      check_bt_error(bt_gemm_splitk_rows(inter_matmul_buf, wt_out, partials, splits, valid_rows, rows, rows_hint,
                                         hidden, inter, weight_kn, stream));
      check_bt_error(bt_splitk_layernorm(
          partials, splits, attr_matmul_buf, nullptr, w.output_bias, w.output_layernorm_gamma,
          w.output_layernorm_beta, use_fp32_ ? 1 : 0,
          restore ? (void *)ip.transformer_output : (void *)ffn2_out,
          restore ? et_param.batch_idx : nullptr, restore ? nullptr : valid_rows, batch_size,
          seq_len, rows, hidden, layernorm_eps, stream));
      continue;
    }
    check_bt_error(bt_gemm(inter_matmul_buf, wt_out, ffn2_out, valid_rows, rows, rows_hint, hidden,
                           inter, weight_kn, stream));
    if (last && is_remove_padding_)
      check_bt_error(bt_add_bias_residual_layernorm_restore(
          ffn2_out, attr_matmul_buf, w.output_bias, w.output_layernorm_gamma,
          w.output_layernorm_beta, use_fp32_ ? 1 : 0, ip.transformer_output, et_param.batch_idx,
          et_param.word_idx, batch_size, seq_len, hidden, layernorm_eps, stream));
    else
      check_bt_error(bt_add_bias_residual_layernorm(
          ffn2_out, attr_matmul_buf, nullptr, w.output_bias, w.output_layernorm_gamma,
          w.output_layernorm_beta, use_fp32_ ? 1 : 0, valid_rows, rows, hidden, layernorm_eps,
          stream));
  }
}

template class BertEncoder<OperationType::FP32>;
template class BertEncoder<OperationType::HALF>;

}  // namespace bytetransformer
