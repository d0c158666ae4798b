// A model: parts built from a ModelSpec, weights loaded into them, and the forward pass of one
// step.  It knows nothing of any architecture: embedding, the blocks in the order the spec gives,
// final norm and head on the wanted rows, as the reference's forward does for its one sequence
// (src/models/turbo_generic.rs:1950-1987).
#pragma once
#include "linear.h"
#include "parts.h"
#include "step.h"
#include "store.h"

namespace tq {

class Model {
public:
    Model(const ModelSpec& spec, int dtype, bool on_gpu);

    ModelSpec spec;
    Json config;                                // the typed configuration it was made from, if any
    int dtype;                                  // F32 or BF16: the run's activation and weight type
    bool on_gpu;                                // false: host memory and no kernels (configuration and weights can still be looked at)
    std::vector<int32_t> stop_token_ids;        // what the configuration names; a model folder may add more
    std::vector<CacheNeed> needs;               // per run of the order
    std::vector<int> cache_of;
    bool graph_safe = false;
    bool loaded = false;

    TensorSpecs tensor_specs() const;
    // Takes the tensors (full names); every part gets its own.  Checks nothing: the loader has.
    void load(Loaded& tensors, hipStream_t stream);
    OwnedPtr held(const std::string& name) const;
    bool head_is_embedding() const { return spec.head_name.empty(); }

    // Runs the step's tokens through every run of the order; logits [wanted rows, vocab] float32 for
    // the step's wanted rows, written to `out` (device memory) or to workspace memory.
    Tensor forward(StepContext& c, const CacheStore& cache, float* out = nullptr);
    // The step in one launch, for small models (small_step.hip): whether that is the way for the planned step, and the step itself.  Nothing
    // of the plan is uploaded: the step's arrays travel with the launch.  device_tokens: as Engine::step.
    // graph_width: the step's tables would be filled up to a multiple of so many pages in a captured graph (1: it would not be captured).
    bool small_step(const StepContext& c, const CacheStore& cache, int graph_width, TqkSmallStep& step) const;
    Tensor forward_small(StepContext& c, TqkSmallStep& step, const int32_t* device_tokens, float* out);
    // Whether a step of that many tokens, decoding or not, up to the furthest position is to be asked about (before anything is planned).
    bool small_pays(long long n_tokens, bool decode, int max_end) const;
    static const int SMALL_ROWS = 64;           // (more rows are not asked about)
    Json describe() const;
    // Lets the library try its kernels once for every product of the model at `rows` rows (more than the own kernels
    // take: fewer never reach the library) and keep the fastest for later calls.
    void tune_library(int64_t rows, hipStream_t stream);

private:
    BuildEnv env_;
    std::vector<std::shared_ptr<Block>> blocks_;
    std::shared_ptr<Norm> final_norm_;
    std::shared_ptr<Position> stream_position_;
    int stream_state_entry_ = -1;               // the cache entry of the stream position's state, if it keeps one
    OwnedPtr embedding_, head_bias_;
    Weight head_;
    bool weights_once_ = false;                 // the weights that steps read whole are more than the memory-side cache holds (256 MB)
    std::unique_ptr<TqkSmallStep> small_;       // the model as that kernel takes it, if it takes any step of it
    void find_small();
    Tensor head_logits(StepContext& c, Stream& stream, float* out);
};

}  // namespace tq
