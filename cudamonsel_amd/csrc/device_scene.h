/*
 * device_scene.h -- device-resident scene layout of the transport engine.
 *
 * The host compiles a monsel_scene_desc (SI, FP64, the reference's object
 * graph) into these flat FP32 records in nm / eV units.  Every record is
 * plain data so that one hipMemcpy uploads the scene.
 */
#ifndef MONSEL_DEVICE_SCENE_H
#define MONSEL_DEVICE_SCENE_H

#include <stdint.h>

/* Scene records are read-only for the lifetime of a kernel, so device code
 * reads them through the constant address space: a load whose index is the
 * same on every lane of a wave then becomes one scalar load into SGPRs
 * instead of a vector load per lane.  (The host pass sees plain pointers of
 * the same size.) */
#if defined(__HIP_DEVICE_COMPILE__)
#define MONSEL_CS __attribute__((address_space(4)))
#else
#define MONSEL_CS
#endif

namespace monsel_dev {

constexpr int kMaxPrims = 8;      /* convex primitives per region shape */
constexpr int kMaxPlanes = 16;    /* planes per multi-plane primitive */
constexpr int kMaxElem = 8;       /* elements per material */
constexpr int kMaxMech = 6;       /* mechanisms per material scatter model */
constexpr int kMaxCore = 8;       /* core levels per material */
constexpr int kMottNE = 61;
constexpr int kMottNQ = 201;

enum PrimKind { PRIM_PLANES = 0, PRIM_CYLINDER = 1, PRIM_SPHERE = 2 };

/* One convex primitive.  Planes: inside is n.p - b <= 0. */
struct DPrim {
  /* 16 words: what a cylinder or a sphere needs, and a multi-plane
   * primitive's counts */
  int kind;
  int n_planes;
  int tie;       /* bit k: a line within plane k counts as inside (plane_tie_break) */
  int first_plane;
  float e0[3];   /* cylinder end0 / sphere centre (nm) */
  float r2;      /* radius^2 (nm^2) */
  float ax[3];   /* cylinder unit axis */
  float len;     /* cylinder length (nm) */
  float sdscale; /* planes: min over the planes of 1/|n| (distance bounds); 1 otherwise */
  float len2;    /* |axv|^2 */
  float pad[2];
  float4 pl[4];  /* the first planes of a multi-plane primitive again, inline (one
                  * fewer dependent load for the common primitives) */
  float axv[3];  /* cylinder axis vector end1-end0 (nm), for point containment */
  float pad2;
};
constexpr int kInlinePlanes = 4;

/* Shapes of at most this many primitives (whose truth table is one 32-bit
 * word) get the sharper safety bound of shape_safety. */
constexpr int kMaxCstPrims = 5;

/* A region shape: a boolean function of up to kMaxPrims primitives, stored
 * as a 256-entry truth table indexed by the primitives' inside bits. */
struct DShape {
  int first_prim;
  int n_prims;
  int is_sphere; /* the chamber sphere: a single primitive */
  int region;    /* the region of this shape, in the list of a region's children */
  uint32_t truth[8];
};

/* JoyLuoNieminenCSD (eV, nm). */
struct DCSD {
  int active;
  int nce;
  float breakE;  /* eV */
  float gamma15; /* 1.5 gamma, 1/(nm eV^1.5) */
  float minE;    /* eV (barrier height) */
  struct Term {  /* one element's; the first three end the record's first 14 words */
    float recipJ; /* 1/eV */
    float beta;
    float coef;   /* eV^2/nm */
  } el[kMaxElem];
  float pad[3];
};

/* One element of an elastic (SelectableElasticSM) mechanism. */
struct DElem {
  float natoms; /* scalefactor * density * N_A, atoms / nm^3 */
  float sfBrowning;
  float brNum;  /* Browning's 3e-4 Z^1.7, 0.005 Z^1.7 and 0.0007 Z^2 */
  float brRoot;
  float brInv;
  int mott;     /* table index or -1 */
  float mottAtMin; /* nm^2 */
  float extrap; /* eV, NISTMottRS extrapolateBelowEnergy (one value per mechanism) */
  int kind;     /* MONSEL_MECH_*_ELASTIC */
  int method;
  float zp3, z;
  float rz13;   /* Z^(1/3) */
  float rz23;   /* Z^(2/3) */
  int Z;
  float pad;
};

/* The elements of an elastic mechanism of at most kFewElem, side by side:
 * what their cross-sections and angles need, read with a few wide scalar
 * loads and evaluated without a loop.  Slots beyond the last element have no
 * atoms. */
constexpr int kFewElem = 3;
struct DFewElem {
  float natoms[kFewElem];
  float sfBrowning[kFewElem];
  float brNum[kFewElem], brRoot[kFewElem], brInv[kFewElem];
  float extrap;          /* eV, NISTMottRS extrapolateBelowEnergy (the elements share it) */
  int spwem[kFewElem];   /* offset of the element's cross-section nodes */
  int x1[kFewElem];      /* and of its angle table */
  float z[kFewElem], zp3[kFewElem];
};

struct DMech {
  int kind;
  int nelem;
  int few;      /* elastic: `el` holds its elements, and their Mott nodes are in LDS */
  int method;
  float extrap; /* elastic: eV, NISTMottRS extrapolateBelowEnergy (its elements share it) */
  int elem0;
  int pad[2];
  float p[24];
  DCSD csd; /* FittedInelSM's slowing-down algorithm */
  DFewElem el;
  int table[4];
  double q[24]; /* tabulated mechanism: the TP_* slots in SI units (J) for the FP64 scatter */
};

/* Tabulated-mechanism parameter slots in DMech::p (eV) and DMech::q (J). */
enum {
  TP_OFFSET = 0, TP_MINEGEN = 1, TP_RATEMULT = 2, TP_E0DISP = 3, TP_CB = 4, TP_BANDGAP = 5,
  TP_GAP = 6, TP_OFFSETFERMI = 7, TP_BEREF = 8, TP_EIDOM0 = 9, TP_EIDOM1 = 10, TP_IIMFPDOM0 = 11,
  TP_IIMFPDOM1 = 12, TP_SE0RANGE0 = 13, TP_SE0RANGE1 = 14, TP_NCORE = 15, TP_CORE0 = 16
};

struct DMSM {
  int is_null;
  int n_mech;
  int mech0;
  int barrier_kind;
  int elastic_k;   /* first elastic mechanism (index within this model), -1 if none */
  int pad[3];
  float minE;      /* eV, may be -inf */
  float cb;        /* eV, material conduction-band bottom */
  float lambdaFactor; /* ExpQMBarrierSM lambda factor, 1/sqrt(eV) */
  float lambda;    /* nm */
  DCSD csd;
};

/* One region.  Its scatter model's and its shape's records are inline, so
 * that a step reads them at an offset of one address. */
struct DRegion {
  DMSM m;
  int parent;
  int msm;
  int first_child;
  int n_children;
  int depth;
  int pad[3];
  DShape sh;
};

/* One axis of a non-uniform table.  The search words (DevScene::nu_words) hold
 * its abscissae (FP64), a guide -- for each bucket of the map below the
 * interval bounds {lo, hi} a point of that bucket lies in -- and for each
 * interval the first point of its cubic window; nu_recs holds a DNUWindow for
 * each interval.  Interval i is between points i and i + 1, i = -1 .. n - 1. */
struct DNUAxis {
  double origin, scale; /* bucket = clamp((v - origin) * scale, 0, last) */
  double last;
  int log;              /* v: the high word of x instead of x */
  int n;
  int x, guide, first;  /* offsets in nu_words: point 0, bucket 0, interval 0 */
  int rec;              /* offset in nu_recs of interval 0 */
  int asc;              /* ascending: bit 0 in FP64, bit 1 rounded to FP32 */
  int pad;
};

/* The x-independent part of the four Lagrange weights over a cubic window. */
struct DNUWindow {
  double x[4];
  double den[4], rden[4]; /* products of differences in units of the span, and 1 / den */
  double inv;             /* 1 / span */
  double pad[3];
};

/* Non-uniform table (NUTableInterpolation) in the file's own units. */
struct DNUTable {
  DNUAxis axis[4];
  int dim;
  int voff;     /* offset of the values, in nu_data (FP32) of a 1-D table, else in nu_data64 */
  int pad[2];
};

struct DevScene {
  int n_regions, n_prims, n_planes, n_msm, n_mech, n_elem, n_mott, n_nu;
  int has_tabulated;      /* some mechanism is TabulatedInelasticSM (selects the transport kernel) */
  uint32_t compat;
  float chamber_r;        /* nm */
  float chamber_c[3];     /* nm */
  const MONSEL_CS DRegion* regions;
  const MONSEL_CS DShape* children;   /* the shapes of each region's children, in a run */
  const MONSEL_CS DPrim* prims;
  const MONSEL_CS float4* planes;   /* (nx, ny, nz, b) */
  const MONSEL_CS DMSM* msms;
  const MONSEL_CS DMech* mechs;
  const MONSEL_CS DElem* elems;
  const MONSEL_CS float* mott_spwem; /* [n_mott][61] */
  const MONSEL_CS float* mott_x1;    /* [n_mott][61*201] */
  const MONSEL_CS DNUTable* nu;
  const MONSEL_CS float* nu_data;
  const MONSEL_CS double* nu_data64;
  const MONSEL_CS unsigned long long* nu_words; /* see DNUAxis */
  const MONSEL_CS DNUWindow* nu_recs;
  int n_nu_words;
};

}  // namespace monsel_dev

#endif
