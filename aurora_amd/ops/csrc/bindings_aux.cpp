// Python bindings of the sentence-encoder, vector-search and collective kernels.
#include <torch/extension.h>

torch::Tensor attention_prefill(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                                torch::Tensor cu, double scale, bool causal);
torch::Tensor attention_prefill_turned(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                                       torch::Tensor cos_sin, torch::Tensor cu, double scale,
                                       bool causal);
torch::Tensor embed_pool(torch::Tensor hidden, torch::Tensor cu);
std::vector<torch::Tensor> knn_topk(torch::Tensor query, torch::Tensor docs, long k);
std::vector<uint8_t> oneshot_init(long world, long rank, long max_bytes);
void oneshot_connect(std::vector<std::vector<uint8_t>> handles);
bool oneshot_ready();
long oneshot_max_bytes();
void oneshot_allreduce_(torch::Tensor t);
void oneshot_destroy();

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("attention_prefill", &attention_prefill, "varlen self-attention (encoder)");
  m.def("attention_prefill_turned", &attention_prefill_turned,
        "the same with queries and keys rotated by their places");
  m.def("embed_pool", &embed_pool, "mean-pool + L2 normalize");
  m.def("knn_topk", &knn_topk, "brute-force kNN top-k");
  m.def("oneshot_init", &oneshot_init, "one-shot allreduce: alloc + IPC handle");
  m.def("oneshot_connect", &oneshot_connect, "one-shot allreduce: map peer buffers");
  m.def("oneshot_ready", &oneshot_ready);
  m.def("oneshot_max_bytes", &oneshot_max_bytes);
  m.def("oneshot_allreduce_", &oneshot_allreduce_, "in-place one-shot xGMI all-reduce (bf16)");
  m.def("oneshot_destroy", &oneshot_destroy);
}
