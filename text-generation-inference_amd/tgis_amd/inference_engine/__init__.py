"""Engine plugin loader: `tgis_amd.inference_engine.<DEPLOYMENT_FRAMEWORK>` must export `InferenceEngine`
(mirrors inference_engine/__init__.py:7-9 of the reference)."""
import importlib


def get_inference_engine_class(deployment_framework: str):
    module = importlib.import_module("tgis_amd.inference_engine." + deployment_framework)
    return module.InferenceEngine
