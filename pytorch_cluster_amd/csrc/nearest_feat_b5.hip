// nearest_feat_impl.hpp for up to 96 components
#include "nearest_feat_impl.hpp"

namespace pca {
PCA_NEAREST_FEAT_DEFINE(5)
PCA_NEAREST_FEAT_DEFINE(6)
} // namespace pca
