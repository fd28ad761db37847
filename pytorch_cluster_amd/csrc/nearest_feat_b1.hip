// nearest_feat_impl.hpp for up to 32 components
#include "nearest_feat_impl.hpp"

namespace pca {
PCA_NEAREST_FEAT_DEFINE(1)
PCA_NEAREST_FEAT_DEFINE(2)
} // namespace pca
