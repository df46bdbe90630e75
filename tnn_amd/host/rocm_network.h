// RocmNetwork: the engine's DefaultNetwork plus, behind a switch, whole-forward graph replay.
//
// On this device the launches of a forward pass are fixed once the instance is initialised (static shapes, stable
// blob and workspace addresses), so after two eager passes - which also perform every lazy allocation - the third can
// be recorded into an executable graph that later calls submit at once (TNN_ROCM_GRAPH=1).  The default is the
// engine's eager layer loop: with the sixty-odd launches a fused encoder is left with, the host stays ahead of the
// device, the gaps between kernels on the device are the same either way, and submitting the recorded graph costs
// more up front than the first eager launch (12-layer encoder, three machines: the replay is 0.5 - 1.8 % slower).
// The replay is for callers whose host thread is slow or busy.  The engine picks the network implementation
// per NetworkType (source/tnn/core/abstract_network.h:102-136, instance.cc:75-85); RocmDevice::ConvertAutoNetworkType()
// names this one, and it registers itself like the engine's other networks (default_network.cc:39-40).
#ifndef TNN_AMD_HOST_ROCM_NETWORK_H_
#define TNN_AMD_HOST_ROCM_NETWORK_H_

#include "rocm_device.h"
#ifdef TNN_ROCM_ENGINE_TREE
#include "tnn/core/default_network.h"
#endif

namespace TNN_NS {

// Layers first .. last of a net that one acc computes in their place.  The graph, its blobs and the memory plan stay those of
// the single layers; what lies between the group's inputs and its output is simply not written.
struct RocmLayerGroup {
    int first = 0, last = 0;
    int projections[3] = {0, 0, 0};    // the layers that make Q, K and V (of an attention core)
    std::shared_ptr<LayerInfo> layer;  // type, inputs, output and parameters of the acc that stands for the group
    std::shared_ptr<LayerResource> resource;
};
// the attention cores (projections included) that an fp32 net keeps as layers
std::vector<RocmLayerGroup> RocmFindAttentionGroups(NetStructure *structure, NetResource *resource);
// the layers that make the masks of a net's attention cores out of integers
std::vector<RocmLayerGroup> RocmFindMaskGroups(NetStructure *structure, NetResource *resource,
                                               const std::vector<RocmLayerGroup> &attention);
// One set of weights for a group and its layers: the attention acc packs the device weights of the three projections, and
// the projections' accs go on with the packed ones.  The attention acc must outlive any Forward of theirs.
Status RocmShareProjections(AbstractLayerAcc *attention, AbstractLayerAcc *const projections[3]);

class RocmNetwork : public DefaultNetwork {
public:
    RocmNetwork();
    ~RocmNetwork() override;
    Status Forward() override;
    Status ForwardAsync(Callback call_back) override;

#ifndef TNN_ROCM_ENGINE_TREE
    Status Init(NetworkConfig &net_config, ModelInterpreter *interpreter, const InputShapesMap &max_inputs_shape = InputShapesMap()) override;
    Status Reshape(const InputShapesMap &inputs) override;

protected:
    // The layer loop of a plain forward.  An fp32 net keeps its attention as layers (every intermediate blob is there for
    // ForwardWithCallback, profiling and whoever names one as a model output), and those ways of running it take them one
    // by one; a plain forward runs each core as a group: one projection for Q, K and V and one attention kernel instead of
    // sixteen launches that pass the [B*h, S, S] scores through memory six times.  In a net of any precision the layers that make
    // the additive mask out of integers are such a group: one launch instead of four (three layers', and the one that takes the
    // key counts from the mask), 12 layers fp16 of 1 x 32 tokens 367 -> 356 us, 1 x 256 481 -> 467, fp32 of 1 x 128 771 -> 753.
    Status RunLayers(void *prof_stream) override;
#endif
#ifdef TNN_ROCM_ENGINE_TREE
protected:
    // The engine settles every blob's data type in UpdateBlobPrecision (default_network.cc:362-440), which returns
    // at once for a device it does not know; this override does that pass for DEVICE_ROCM and then runs the engine's
    // own InitLayers.
    Status InitLayers(NetStructure *net_structure, NetResource *net_resource) override;
#if TNN_PROFILE
    Status ProfiledForward();  // the forward loop with every layer timed (a profiler build of the engine)
#endif
#endif

private:
#ifndef TNN_ROCM_ENGINE_TREE
    struct Group {
        int first = 0, last = 0;
        bool active = false;  // false: the shapes or the memory plan at hand do not allow it, its layers run one by one
        std::shared_ptr<LayerInfo> layer;
        std::shared_ptr<LayerResource> resource;
        std::unique_ptr<AbstractLayerAcc> acc;
        std::vector<Blob *> inputs, outputs;
    };
    Status ReshapeGroups();
    std::vector<Group> groups_;
#endif
    // Everything a recording depends on: dims and device address of every blob the layers touch, the context's scratch
    // allocation count and the form of the result stores.  A recording is replayed only under the signature it was made with, so a Reshape, a
    // re-planned blob pool or a grown workspace lead back to eager passes and a new recording by themselves.
    void Signature(std::vector<uint64_t> *sig);
    void DropGraphs();
    void DropProfileEvents();
    std::vector<void *> profile_events_;  // two per layer, created at the first profiled forward
    struct Recording {
        std::vector<uint64_t> signature;
        void *exec = nullptr;
    };
    std::vector<Recording> recordings_;
    std::vector<uint64_t> eager_signature_;
    int eager_forwards_ = 0;
    bool enabled_       = false;  // TNN_ROCM_GRAPH=1 turns the replay on; the default is the engine's eager loop
};

}  // namespace TNN_NS
#endif
