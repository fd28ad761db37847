// nearest_feat_impl.hpp for up to 128 components
#include "nearest_feat_impl.hpp"

namespace pca {
PCA_NEAREST_FEAT_DEFINE(7)
PCA_NEAREST_FEAT_DEFINE(8)
} // namespace pca
