// model_runner.h -- the decode loop of AsModel for DeviceType::HIP, reduced to what drives the hot path:
//   context phase   AsModel::runDecoderContext (csrc/core/model/model.cpp:566-650): one request, Reshape -> Alloc -> Forward
//   decoder phase   AsModel::GenerateContinueDecoder (model.cpp:1212-1325): the running batch, Reshape only when the batch
//                   membership changed, Alloc -> Forward per operator per step
// over an operator list built through OpFactory (model.cpp:265-287) -- the reference graph as it is, or rewritten by
// host/fusion_pass.cpp into the fused decode-step operators.  With the fused list the decoder phase keeps its whole state on the
// device (next input ids, sequence lengths, span tables), so that a step is a pure function of device memory and is captured
// ONCE into a hipGraph and replayed (hipGraphLaunch per step); the host only claims cache spans (CallAlloc) and counts steps.
// Not here (the reference's own, device-independent): scheduler, request queues, stop conditions, tokenizer, weight loading.
#pragma once
#include <memory>
#include <string>
#include <vector>

#include "fusion_pass.h"
#include "operator.h"

namespace allspark {

class HipModelRunner {
 public:
  HipModelRunner(HIPContext* ctx, TensorMap* tensors, TensorMap* weights, TensorMap* weights_buffer);
  ~HipModelRunner();

  // graph: the reference's operator list in execution order (first operator reads the id tensor, last one writes the ids)
  AsStatus Build(const std::vector<OperatorProto>& graph, bool fuse);
  const FusionReport& fusion() const { return fusion_; }
  const std::vector<OperatorProto>& protos() const { return protos_; }

  // A request enters through its context phase: prompt ids on the host, its GenerateContext (caches, prefix_len, gen_cfg).
  // Runs eagerly; *first_id = the token sampled after the prompt.  The request then joins the running batch.
  AsStatus StartRequest(std::shared_ptr<GenerateContext> gc, const int64_t* prompt_host, int len, int64_t* first_id);
  // A request whose cache already holds gc->step tokens joins the batch with `next_id` as its next input (benchmarks)
  AsStatus AdoptRequest(std::shared_ptr<GenerateContext> gc, int64_t next_id);
  AsStatus StopRequest(int index);
  int batch() const { return (int)running_.size(); }
  const std::vector<std::shared_ptr<GenerateContext>>& running() const { return running_; }

  // What the next decoder step of the running batch needs before it can be launched, if it is not there yet: operators reshaped for the batch (tensors grow: hipMalloc, and
  // hipFree, which waits for all work on the device), the step captured and instantiated.  DecodeSteps does it by itself; ranks that share one GPU and wait for one another in
  // their all-reduces all go through this first, then launch -- a rank that still frees memory would wait for a peer's all-reduce, which waits for this rank.
  AsStatus PrepareDecode(bool use_graph);
  // n decoder steps of the running batch.  use_graph: capture the step once, replay it (fused list only)
  AsStatus DecodeSteps(int n, bool use_graph);
  // Benchmarks: every running request back to `cached_len` tokens (the caller rewinds the requests' caches; the span tables and
  // the captured step stay as they are -- no operator is reshaped): lengths re-uploaded, next ids kept.
  AsStatus Rewind(int cached_len);
  // stream synchronise + the ids generated by the last step, one per running request
  AsStatus Sync(std::vector<int64_t>* ids);
  const std::string& last_error() const { return err_; }
  // the last Sync failed on the fused attention block's error word, or the peer-to-peer communicator's: the running requests' gen_ctx->step are back at the last good
  // synchronise and next ids are that synchronise's; the OWNER of the virtual caches rewinds them to gen_ctx->step (or fails the requests)
  bool handoff_failed() const { return handoff_failed_; }

 private:
  AsStatus PrepareBatch();
  AsStatus Fail(AsStatus st, const std::string& what);
  AsStatus ForEach(RuntimeContext* rt, int phase);  // 0 Reshape, 1 Alloc, 2 Forward
  void BindIds(void* data, int64_t rows, int64_t cols);
  void DropGraph();

  HIPContext* ctx_;
  TensorMap *tensors_, *weights_, *weights_buffer_;
  std::vector<OperatorProto> protos_;
  std::vector<std::unique_ptr<AsOperator>> ops_;
  FusionReport fusion_;
  std::string ids_in_name_, ids_out_name_, err_;
  RuntimeContext decode_rt_;
  std::vector<std::shared_ptr<GenerateContext>> running_;
  std::vector<int64_t> next_ids_;
  bool dirty_ = true, fused_ = false;
  std::unique_ptr<AsTensor> prompt_dev_;
  int64_t* ids_pinned_ = nullptr;   // [max_batch] staging up, [max_batch] staging down
  int32_t* lens_pinned_ = nullptr;  // [2 * max_batch]
  bool handoff_failed_ = false;            // the last Sync failed on the attention block's or the all-reduce's error word: requests rolled back (gen_ctx->step), caches are the owner's to rewind
  int steps_since_sync_ = 0;               // decode steps enqueued since the last successful Sync (rolled back when the block's error word is set)
  unsigned* block_err_pinned_ = nullptr;  // the fused attention block's error word, read back with the ids (Sync)
  int64_t* prompt_pinned_ = nullptr;
  size_t prompt_cap_ = 0;
  hipEvent_t staged_ = nullptr;
  hipGraph_t graph_ = nullptr;
  hipGraphExec_t graph_exec_ = nullptr;
};

}  // namespace allspark
