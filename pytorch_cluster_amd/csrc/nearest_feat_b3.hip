// nearest_feat_impl.hpp for up to 64 components
#include "nearest_feat_impl.hpp"

namespace pca {
PCA_NEAREST_FEAT_DEFINE(3)
PCA_NEAREST_FEAT_DEFINE(4)
} // namespace pca
