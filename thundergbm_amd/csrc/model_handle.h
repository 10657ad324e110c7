// The model handle of the C ABI (`Tree*&` in the reference's scikit_tgbm.cpp): all trees, iteration-major, the
// class trees of an iteration next to each other. Opaque to callers; shared by the translation units that
// implement entry points taking a handle. The trees never change once the handle exists.
#pragma once
#include <memory>
#include <mutex>
#include <vector>

#include "host.h"

namespace tgbm {
struct DeviceModel;  // predictor.hip: the model as the scoring kernels read it, on one GPU
}

struct tgbm_model {
    std::vector<tgbm::Tree> trees;
    // Laid out by the first call that scores with the handle and kept until model_free; laid out anew for another GPU or
    // another number of trees. Calls hold a reference while they use it.
    std::mutex mutex;
    std::shared_ptr<const tgbm::DeviceModel> on_device;
};

namespace tgbm {

// Predictor::predict_raw / predict (src/thundergbm/predictor.cu:11-189) with the first n_iter x n_class trees of the
// handle. out: class-major raw scores (n rows x n_class floats), or with `transform` the objective's predictions.
void score(const GBMParam &param, tgbm_model &model, int n_iter, int n_class, const DataSet &ds, bool transform,
           bool log_metric, float *out);

}  // namespace tgbm
