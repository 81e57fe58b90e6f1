// acnet.hpp -- the reference actor-critic's minibatch (one latent-attention layer, d 64) as one
// kernel (acnet.hip), used by the PPO plan where acnet_supported holds.
#pragma once

#include "common.hpp"

namespace talos {

struct AcNetCall {
  int n = 0;  // samples
  const float* params = nullptr;
  const float* states = nullptr;
  const int32_t* lens = nullptr;
  const float* rcos = nullptr;  // [seq][8]
  const float* rsin = nullptr;
  // forward only: [n][A], [n] (either may be null)
  float* logits = nullptr;
  float* values = nullptr;
  // minibatch
  const int32_t* actions = nullptr;
  const float* adv = nullptr;
  const float* ret = nullptr;
  const float* old_logp = nullptr;
  float* loss = nullptr;     // may be null
  float* dparams = nullptr;
  double* stats = nullptr;   // may be null
  int stats_acc = 0;
  double* ws = nullptr;  // acnet_ws_bytes
};

// Whether the network is the reference actor-critic's shape (ActorCritic::new, src/ppo.rs:254-258):
// in_dim 8, d 64, one latent-attention layer of 4 heads (latent 32, rope 16, head and value dims
// 16), ffn 128, at most 8 actions, seq <= 128.
bool acnet_supported(const talos_ppo_cfg& c);
// The most workspace a call needs (the workgroups' gradient partials), for num_cu CUs.
size_t acnet_ws_bytes(const talos_ppo_cfg& c, int num_cu);
int acnet_forward_launch(const talos_ppo_cfg& c, int num_cu, const AcNetCall& a, hipStream_t s);
int acnet_minibatch_launch(const talos_ppo_cfg& c, int num_cu, const AcNetCall& a, hipStream_t s);

}  // namespace talos
