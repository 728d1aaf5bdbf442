/*
 * ixt_train.h -- C ABI of the training step of libixt.so: forward + backward of the
 * llama2 block stack on one GPU's share of the batch, cross entropy with the reference's custom VJP, global-norm clip and AdamW.
 * Same boundary rules as ixt.h: plain C, int status, explicit stream, no allocation after create.  Parameters, gradients and the AdamW
 * moments live in FLAT f32 device buffers owned by the CALLER, laid out as ixt_train_param_info describes, so that the data-parallel
 * exchange (RCCL reduce-scatter + all-gather over xGMI, driven by torch.distributed in maxtext-indextts2_amd/train.py) runs on them in place.
 * Each entry point names the reference code it stands for (paths relative to the reference repo).
 */
#ifndef IXT_TRAIN_H_
#define IXT_TRAIN_H_

#include "ixt.h"

#ifdef __cplusplus
extern "C" {
#endif

typedef struct ixt_train_config {
  int32_t vocab_size, emb_dim, num_query_heads, num_kv_heads, head_dim, mlp_dim, num_decoder_layers;   /* as ixt_config */
  float normalization_layer_epsilon, rope_min_timescale, rope_max_timescale;
  int32_t batch;          /* rows of this GPU's batch = per_device_batch_size (train.py:271-275) */
  int32_t seq_len;        /* max_target_length (base.yml:527) */
  int32_t logits_chunk;   /* rows whose [rows, vocab] logits (bf16) and their gradients are alive at a time (0: 2048).  rows x vocab f32 words are set aside
                             for them, which the backward pass uses for the parts of long reductions */
} ixt_train_config;

typedef struct ixt_trainer ixt_trainer;

const char* ixt_train_last_error(void);
/* maxtext_utils.setup_training_state (state shapes) + activation workspaces for one batch of [batch, seq_len]. */
int ixt_train_create(const ixt_train_config* cfg, ixt_trainer** out);
/* The same with a say in how attention goes: IXT_TRAIN_ATTENTION_AUTO is ixt_train_create; _WALK: scores, softmax and products in one launch (head_dim 64 or 128, seq_len at
 * most 4096; IXT_ERR_UNSUPPORTED elsewhere); _MEMORY: one behind the other, through memory (any size). */
#define IXT_TRAIN_ATTENTION_AUTO 0
#define IXT_TRAIN_ATTENTION_WALK 1
#define IXT_TRAIN_ATTENTION_MEMORY 2
int ixt_train_create_attention(const ixt_train_config* cfg, int attention, ixt_trainer** out);
int ixt_train_destroy(ixt_trainer* t);
/* The flat parameter layout: `count` tensors, tensor i = `numel` f32 values at `offset` (elements) of the flat buffers, row-major with
 * MaxText's kernel shapes; `name` is the unscanned tree path ("params/decoder/layers_3/mlp/wi_0/kernel"). */
int64_t ixt_train_total_numel(ixt_trainer* t);
int ixt_train_param_count(ixt_trainer* t);
int ixt_train_param_info(ixt_trainer* t, int index, char* name_out, int name_cap, int64_t* offset, int64_t* numel);
/* Caller-owned flat f32 device buffers of ixt_train_total_numel elements each: TrainState.params, the gradient tree, AdamW mu and nu. */
int ixt_train_bind(ixt_trainer* t, float* params, float* grads, float* adam_mu, float* adam_nu);
/* bf16 compute copies of the parameters (linears.py:216: kernels are cast to the activation dtype at use); call after loading params. */
int ixt_train_refresh_bf16(ixt_trainer* t, void* stream);
/* train.loss_fn + jax.value_and_grad (train.py:255-351, :415-416) on this GPU's rows: int32 [batch, seq_len] device arrays with the six-key
 * batch contract (maxtext_utils.py:85-99; targets_position is not needed).  Writes loss_and_weights_dev = {total_loss = sum of xent over
 * weighted positions, total_weights} (f32[2], :307-309) and the gradient of total_loss into the bound gradient buffer (overwritten). */
int ixt_train_forward_backward(ixt_trainer* t, const int32_t* inputs, const int32_t* inputs_position, const int32_t* inputs_segmentation,
                               const int32_t* targets, const int32_t* targets_segmentation, float* loss_and_weights_dev, void* stream);
/* The rest of train_step on the (already data-parallel-reduced) gradient buffer: divide by total_weights + EPS (:322), clip by global
 * norm (maxtext_utils.py:825-846, optax.clip_by_global_norm), optax.adamw update number `count` (1-based; optimizers.py:28-38), refresh of
 * the bf16 copies.  norms_out_dev f32[2] = {raw_grad_norm, grad_norm} (train.py:457-458). */
int ixt_train_apply(ixt_trainer* t, float total_weights, float clip_threshold, float lr, float b1, float b2, float eps, float eps_root,
                    float weight_decay, int count, float* norms_out_dev, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* IXT_TRAIN_H_ */
