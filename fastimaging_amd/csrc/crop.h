// Index rules of the cropped image store of the c2r (fft.hip): from the rows of a padded
// column to the rows of the image column and to the entries of the correction table.
// Plain C++, so that the host can check them too.
#pragma once

#ifdef __HIPCC__
#define STP_HD __host__ __device__ __forceinline__
#else
#define STP_HD inline
#endif

namespace stp_hip {

// Image row that row y of a padded column of n rows becomes, or -1 where it is cropped
// away (normalise_image_beam_result_1D, imager.h:99-150).
STP_HD int crop_row(int y, int n, int img)
{
    const int hi = img / 2;
    return y < hi ? y : y >= n - (img - hi) ? y - n + img : -1;
}

// Entry of image row i in a table with row 0's entry at 0, in [-n/2, n/2) whatever i is:
// a cropped row (-1), whose value goes unused, takes row 0's, so that the loads of a pair
// need no branch.
STP_HD int crop_table_at(int i, int img)
{
    const int k = i < 0 ? 0 : i;
    return k < img / 2 ? k : k - img;
}

// Rows ya and yb of a padded column in the image: their rows, and whether both are stored as
// one pair.
struct CropPair {
    int ia, ib;
    bool pair;
};
STP_HD CropPair crop_pair(int ya, int yb, int n, int img)
{
    const int ia = crop_row(ya, n, img), ib = crop_row(yb, n, img);
    return { ia, ib, ia >= 0 && ib == ia + 1 };
}

} // namespace stp_hip
